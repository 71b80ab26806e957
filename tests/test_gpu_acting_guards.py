"""Acting steps on parameters and inputs as programs have them: views into flat vectors, hooks, second names."""
import pytest
import torch

from memorax_amd import sequence_models as sm
from memorax_amd._lib import native

pytestmark = pytest.mark.gpu

CELLS = {"lru": lambda: sm.LRUCell(64, 64), "mamba": lambda: sm.MambaCell(64, num_heads=2, head_dim=16, state_dim=16),
         "mlstm": lambda: sm.mLSTMCell(64, hidden_dim=64, num_heads=2), "linear_attention": lambda: sm.LinearAttentionCell(64, 16, 2),
         "delta": lambda: sm.DeltaNetCell(64, 16, 2)}


def _block(cell):
    torch.manual_seed(0)
    with torch.device("cuda"):
        return sm.Residual(sm.PreNorm(sm.Memoroid(CELLS[cell]()), 64)).cuda()


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("cell", sorted(CELLS))
def test_parameters_off_their_boundaries(cell, T):
    """Parameters that are views into a vector at odd offsets, a misaligned input: the same numbers."""
    block = _block(cell)
    x, done = torch.randn(6, T, 64, device="cuda"), torch.zeros(6, T, dtype=torch.bool, device="cuda")
    with torch.no_grad():
        want = block(x, done)[1]
        for name, p in block.named_parameters():
            if T > 1 and "norm" in name:   # the norm kernels over whole rollouts take aligned parameters only
                continue
            flat = torch.empty(p.numel() + 1, device="cuda", dtype=p.dtype)
            flat[1:] = p.flatten()
            p.data = flat[1:].view(p.shape)
        if T == 1:
            flat = torch.empty(x.numel() + 1, device="cuda")
            flat[1:] = x.flatten()
            x = flat[1:].view(x.shape)
        got = block(x, done)[1]
    # the same kernels or the array library's products in another order of summation: float32 sums of 64 terms, bfloat16 for delta
    torch.testing.assert_close(got, want, rtol=0, atol=2e-2 if cell == "delta" else 1e-5 * float(want.abs().max()))


@pytest.mark.parametrize("cell", sorted(CELLS))
def test_a_hook_runs(cell):
    block = _block(cell)
    seen = []
    block.module.module.cell.register_forward_hook(lambda m, i, o: seen.append(1))
    with torch.no_grad():
        block(torch.randn(6, 1, 64, device="cuda"), torch.zeros(6, 1, dtype=torch.bool, device="cuda"))
    assert seen


PARTS = {"lru": ["", "cell"], "mamba": ["", "cell", "cell.output_projection"], "mlstm": ["", "cell", "cell.output_projection"],
         "linear_attention": ["", "cell.norm", "cell.output_projection"], "delta": ["", "cell.output_projection"], "recurrence": ["", "out"]}


@pytest.mark.parametrize("T,grad", [(1, False), (5, False), (5, True)])
@pytest.mark.parametrize("cell,part,autocast", [(c, p, a) for c in sorted(PARTS) for p in PARTS[c] for a in (False, True)
                                                if not (a and c == "mamba")])   # (float32 only)
def test_a_forward_set_on_an_instance_runs(cell, part, autocast, T, grad):
    """As adapters and accelerators set it: on a layer, a cell or the sequence model, acting and over sequences."""
    block = _block(cell) if cell in CELLS else sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(64), 64)).cuda()
    m, seen = block.module.module.get_submodule(part), []
    own = m.forward
    m.forward = lambda *a, **k: seen.append(1) or own(*a, **k)
    with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        block(torch.randn(6, T, 64, device="cuda"), torch.zeros(6, T, dtype=torch.bool, device="cuda"))
    assert seen


@pytest.mark.parametrize("dual", ["input", "parameter", "carry"])
@pytest.mark.parametrize("cell", [*sorted(CELLS), "recurrence"])
def test_an_acting_block_refuses_tangents(cell, dual):
    block = _block(cell) if cell in CELLS else sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(64), 64)).cuda()
    x, done = torch.randn(6, 1, 64, device="cuda"), torch.zeros(6, 1, dtype=torch.bool, device="cuda")
    carry = block.initialize_carry(None, (6, 64))
    make = lambda t: torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))  # noqa: E731
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        params = {}
        if dual == "input":
            x = make(x)
        elif dual == "carry":
            carry = (make(carry[0]), *carry[1:])
        else:
            name, p = next((n, p) for n, p in block.named_parameters() if p.dim() == 2)
            params[name] = make(p.detach())
        with pytest.raises(NotImplementedError, match="forward-mode"):
            torch.func.functional_call(block, params, (x, done, carry))


@pytest.mark.parametrize("dual", ["input", "flags", "carry"])
@pytest.mark.parametrize("cell", ["delta", "linear_attention", "recurrence"])
def test_an_acting_stack_refuses_tangents(cell, dual):
    block = _block(cell) if cell in CELLS else sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(64), 64)).cuda()
    stack = sm.Stack([block, sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(64), 64)).cuda()])
    x, done, carry = torch.randn(6, 1, 64, device="cuda"), torch.zeros(6, 1, device="cuda"), stack.initialize_carry(None, (6, 64))
    make = lambda t: torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))  # noqa: E731
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        x, done = make(x) if dual == "input" else x, make(done) if dual == "flags" else done
        if dual == "carry":
            carry = (carry[0], (make(carry[1][0]), carry[1][1]))
        with pytest.raises(NotImplementedError, match="forward-mode"):
            stack(x, done, carry)


@pytest.mark.parametrize("cell", ["lru", "mlstm", "recurrence"])
def test_blocks_wider_than_the_row_kernel_act_on_their_composition(cell):
    Fe = 2056
    torch.manual_seed(1)
    make = {"lru": lambda: sm.Memoroid(sm.LRUCell(Fe, 16)), "mlstm": lambda: sm.Memoroid(sm.mLSTMCell(Fe, hidden_dim=32, num_heads=2)),
            "recurrence": lambda: sm.GatedLinearRecurrence(Fe, 16)}[cell]
    block = sm.Residual(sm.PreNorm(make(), Fe, norm=sm.RMSNorm)).cuda()
    x, done = torch.randn(3, 1, Fe, device="cuda"), torch.zeros(3, 1, dtype=torch.bool, device="cuda")
    with torch.no_grad():
        y = block(x, done)[1]
    want = block(x, done)[1]
    torch.testing.assert_close(y, want, rtol=0, atol=1e-5 * float(want.detach().abs().max()))


@pytest.mark.parametrize("part", ["cell.z", "cell.h", "gate", "out"])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("autocast", [False, True])
def test_a_layer_left_on_the_host_is_an_error(part, first, autocast):
    """Before a launch has its address; the first step (no carry yet) and one that carries on."""
    block = sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(64), 64)).cuda()
    carry = None if first else block.initialize_carry(None, (6, 64))
    block.module.module.get_submodule(part).cpu()
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        with pytest.raises(ValueError, match="must live on the GPU"):
            block(torch.randn(6, 1, 64, device="cuda"), torch.zeros(6, 1, dtype=torch.bool, device="cuda"), carry)


@pytest.mark.parametrize("at", ["scale", "weight", "closing weight", "bias", "done", "log_state", "log_decay"])
def test_whatever_a_gated_step_reads_is_on_its_gpu(at):
    x, done, ones = torch.randn(6, 1, 64, device="cuda"), torch.zeros(6, 1, device="cuda"), torch.ones(64, device="cuda")
    ws, bs, state = [torch.randn(64, 64, device="cuda") for _ in range(4)], [None] * 4, torch.zeros(6, 1, 64, device="cuda")
    host = lambda t, name: t.cpu() if at == name else t  # noqa: E731
    ws[1], ws[3], bs[0] = host(ws[1], "weight"), host(ws[3], "closing weight"), ones.cpu() if at == "bias" else None
    with torch.no_grad(), pytest.raises(ValueError, match="must live on the GPU"):
        native().gated_act(x, 1, host(ones, "scale"), None, 1e-6, ws, bs, torch.float32, host(done, "done"), host(state, "log_state"),
                           host(state.clone(), "log_decay"), False)


def _counting(cls, method, seen):
    """A subclass of ``cls`` that notes each call of ``method``."""
    def run(self, *a, **k):
        seen.append(1)
        return getattr(cls, method)(self, *a, **k)
    return type("Own" + cls.__name__, (cls,), {method: run})


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("replaced", ["memoroid", "recurrence cell scan", "recurrence cell elements", "mamba conv", "mlstm conv"])
def test_a_subclass_runs_what_it_overrides(replaced, T):
    seen = []
    if replaced == "memoroid":
        model = _counting(sm.Memoroid, "forward", seen)(sm.LinearAttentionCell(64, 16, 2))
    elif "conv" in replaced:
        cell = CELLS[replaced.split()[0]]()
        name = "conv" if replaced.startswith("mamba") else "causal_conv"
        old = getattr(cell, name)
        setattr(cell, name, _counting(torch.nn.Conv1d, "forward", seen)(old.in_channels, old.out_channels, 4, groups=old.groups))
        model = sm.Memoroid(cell)
    else:
        model = sm.GatedLinearRecurrence(64)
        model.cell = _counting(sm.MinGRUCell, replaced.split()[-1], seen)(64)
    block = sm.Residual(sm.PreNorm(model, 64)).cuda()
    with torch.no_grad():
        block(torch.randn(6, T, 64, device="cuda"), torch.zeros(6, T, dtype=torch.bool, device="cuda"))
    assert seen


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("cell,make", [("mamba", lambda c: torch.nn.Conv1d(c, c, 4, groups=c, bias=False)), ("mlstm", lambda c: torch.nn.Conv1d(c, c, 4)),
                                       ("mlstm", lambda c: torch.nn.Conv1d(c, c, 4, groups=c, bias=False))])
def test_convolutions_that_are_no_causal_kernel_s(cell, make, T):
    """Without a bias, or over every channel: the array library's, in both directions."""
    block = _block(cell)
    inner = block.module.module.cell
    name = "conv" if cell == "mamba" else "causal_conv"
    setattr(inner, name, make(getattr(inner, name).in_channels).cuda())
    x, done = torch.randn(6, T, 64, device="cuda"), torch.zeros(6, T, dtype=torch.bool, device="cuda")
    with torch.no_grad():
        got = block(x, done)[1]
    want = block(x, done)[1]
    want.sum().backward()
    assert getattr(inner, name).weight.grad is not None
    torch.testing.assert_close(got, want, rtol=0, atol=1e-5 * float(want.detach().abs().max()))


@pytest.mark.parametrize("T,grad", [(1, False), (5, False), (5, True)])
@pytest.mark.parametrize("norm", [sm.RMSNorm, sm.LayerNorm])
@pytest.mark.parametrize("way", ["hook", "instance", "subclass"])
@pytest.mark.parametrize("part", ["block", "norm"])
def test_a_pre_norm_block_around_the_fork_runs_what_was_put_in(part, way, norm, T, grad):
    """x + f(norm(x)) through the norm's two results passes neither the norm nor the block around it by."""
    seen = []
    block = sm.PreNorm(sm.GatedLinearRecurrence(64), 64, norm=norm)
    if way == "subclass" and part == "norm":
        cls = type(block.norm)
        block.norm = _counting(cls, "forward", seen)(64)
    elif way == "subclass":
        block = _counting(sm.PreNorm, "forward", seen)(block.module, 64, norm=norm)
    m = block if part == "block" else block.norm
    if way == "hook":
        m.register_forward_hook(lambda *a: seen.append(1))
    elif way == "instance":
        own = m.forward
        m.forward = lambda *a, **k: seen.append(1) or own(*a, **k)
    with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.bfloat16):
        sm.Residual(block).cuda()(torch.randn(6, T, 64, device="cuda"), torch.zeros(6, T, dtype=torch.bool, device="cuda"))
    assert seen
