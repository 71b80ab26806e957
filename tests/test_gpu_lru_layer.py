"""The LRU cell's layer as one operation (csrc/lru_cells.hip, native().lru_layer) against float64 and against its composition; the float32
closing layers that add to the residual stream."""
import pytest
import torch

from memorax_amd import _lib
from memorax_amd import sequence_models as sm

pytestmark = pytest.mark.gpu


def _err(a, b):
    return float(((a.detach() - b).abs().norm() / b.abs().norm().clamp_min(1e-300)))


def _float64(cell, x, done, h0):
    """The recurrence step by step (lru.py:76-108)."""
    p = {k: v.detach().double().requires_grad_() for k, v in cell.named_parameters()}
    x, h0 = x.detach().double().requires_grad_(), h0.detach().to(torch.complex128).requires_grad_()
    lam = torch.polar(torch.exp(-torch.exp(p["nu_log"])), torch.exp(p["theta_log"]))
    u = torch.complex(x @ p["B_real"].t(), x @ p["B_imag"].t()) * torch.exp(p["gamma_log"])
    h, states = h0, []
    for t in range(x.shape[1]):
        h = torch.where(done[:, t, None], u[:, t], lam * h + u[:, t])
        states.append(h)
    y = (torch.stack(states, 1) @ torch.complex(p["C_real"], p["C_imag"]).t()).real + p["D"] * x
    return y, h, x, h0, p


@pytest.mark.parametrize("B,T,F,N", [(8, 8, 64, 32), (13, 5, 64, 36), (33, 50, 128, 128), (600, 20, 72, 100), (64, 64, 256, 256)])
def test_layer_against_float64(B, T, F, N):
    """No further from float64 than the composition, up to a tenth and a rounding of the result."""
    torch.manual_seed(B)
    print(f"case lru layer {B} {T} {F} {N}", flush=True)
    cell = sm.LRUCell(F, N).cuda()
    x, done = torch.randn(B, T, F, device="cuda").requires_grad_(), torch.rand(B, T, device="cuda") < 0.05
    h0, P0 = torch.randn(B, 1, N, dtype=torch.complex64, device="cuda").requires_grad_(), torch.ones(B, 1, N, dtype=torch.complex64, device="cuda")
    gy, gh = torch.randn(B, T, F, device="cuda"), torch.randn(B, N, dtype=torch.complex64, device="cuda")
    y64, h64, x64, h064, p64 = _float64(cell, x, done, h0[:, 0])
    torch.autograd.backward([y64, h64], [gy.double(), gh.to(torch.complex128)])

    def errors(run):
        for t in (x, h0, *cell.parameters()):
            t.grad = None
        carry, y = run()
        torch.autograd.backward([y, carry[0][:, 0]], [gy, gh])
        return [_err(y, y64), _err(carry[0][:, 0], h64), _err(x.grad, x64.grad), _err(h0.grad[:, 0], h064.grad),
                *(_err(p.grad, p64[k].grad) for k, p in cell.named_parameters())], carry

    def composition():
        h, carry = cell.scan(cell(x), (h0, P0), done)
        return carry, cell.read(h, x)

    assert cell.whole(x, done, (h0, P0)) is not None
    (here, carry), (there, ref) = errors(lambda: cell.whole(x, done, (h0, P0))), errors(composition)
    assert all(a <= 1.1 * b + 2.0 ** -23 for a, b in zip(here, there)), (here, there)
    assert [c.shape for c in carry] == [c.shape for c in ref] and torch.allclose(carry[1], ref[1], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("cell", ["lru", "mamba", "linear_attention", "recurrence"])
def test_blocks_on_a_float32_stream(cell):
    """Residual(PreNorm(model)): the sum with the stream inside the closing layer, against the sum behind it; float32 sums of up to 128 terms."""
    torch.manual_seed(3)
    make = {"lru": lambda: sm.Memoroid(sm.LRUCell(64, 64)), "mamba": lambda: sm.Memoroid(sm.MambaCell(64, num_heads=2, head_dim=32, state_dim=16)),
            "linear_attention": lambda: sm.Memoroid(sm.LinearAttentionCell(64, 32, 2)), "recurrence": lambda: sm.GatedLinearRecurrence(64)}[cell]
    block = sm.Residual(sm.PreNorm(make(), 64)).cuda()
    x, done = torch.randn(9, 40, 64, device="cuda"), torch.rand(9, 40, device="cuda") < 0.05
    g = torch.randn_like(x)

    def run(forward):
        xs = x.clone().requires_grad_()
        block.zero_grad(set_to_none=True)
        _, y = forward(xs)
        y.backward(g)
        return [y.detach(), xs.grad, *(p.grad.clone() for p in block.parameters())]

    inner = block.module

    def behind(xs):
        carry, y = inner.module(inner.norm(xs), done, None)
        return carry, xs + y

    for a, b in zip(run(lambda xs: block(xs, done)), run(behind)):
        assert _err(a.double(), b.double()) <= 2e-5


@pytest.mark.parametrize("cell", ["lru", "lru of few rows", "s5", "mamba", "linear_attention", "recurrence"])
def test_a_block_makes_its_carry_once(cell):
    """Whether the closing layer takes the sum with the stream, or the block finds that it does not."""
    make = {"lru": lambda: sm.Memoroid(sm.LRUCell(64, 64)), "s5": lambda: sm.Memoroid(sm.S5Cell(64, 32)),
            "mamba": lambda: sm.Memoroid(sm.MambaCell(64, num_heads=2, head_dim=32, state_dim=16)),
            "linear_attention": lambda: sm.Memoroid(sm.LinearAttentionCell(64, 32, 2)), "recurrence": lambda: sm.GatedLinearRecurrence(64)}[cell.split(" of")[0]]
    block = sm.Residual(sm.PreNorm(make(), 64)).cuda()
    rows, steps, inner = 3 if "few" in cell else 9, 20, block.module.module.cell
    made, init = [], type(inner).initialize_carry

    class Counting(type(inner)):
        def initialize_carry(self, key, input_shape):
            made.append(input_shape)
            return init(self, key, input_shape)

    inner.__class__ = Counting
    x, done = torch.randn(rows, steps, 64, device="cuda"), torch.rand(rows, steps, device="cuda") < 0.05
    block(x.requires_grad_(), done)
    assert len(made) == 1


def test_saved_tensors_in_another_layout():
    """A hook on saved tensors may hand them back with other strides."""
    torch.manual_seed(4)
    cell = sm.LRUCell(64, 32).cuda()
    x, done = torch.randn(8, 16, 64, device="cuda").requires_grad_(), torch.zeros(8, 16, device="cuda", dtype=torch.bool)
    carry = cell.initialize_carry(None, (8, 64))

    def grads():
        _, y = cell.whole(x, done, carry)
        return torch.autograd.grad(y.square().sum(), [x, *cell.parameters()])

    want = grads()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.t().contiguous().t() if t.dim() == 2 else t):
        got = grads()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("rows,D", [(1, 1), (63, 64), (65, 65), (8192, 72), (20011, 256)])
def test_column_product(rows, D):
    import ctypes
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(rows)
    a, b = (torch.randn(rows, D, device="cuda", generator=g) for _ in range(2))
    out = torch.empty(D, device="cuda")
    work = torch.empty(max(1, lib.mrx_column_product_workspace(rows, D)), device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert lib.mrx_column_product(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ptr(a), ptr(b), ptr(out), ptr(work), rows, D) == 0
    want = (a.double() * b.double()).sum(0)
    # chains of rows / 128 / 64 additions, partial sums in pairs: a few roundings of the products' 2-norm
    assert ((out.double() - want).abs() <= 16 * 2.0 ** -24 * (a.double() * b.double()).norm(dim=0)).all()
