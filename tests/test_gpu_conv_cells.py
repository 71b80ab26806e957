"""The Mamba cell as one operation (MambaCell.whole: conv_cells.hip around the gated kernels) against the cell's own
composition of array operations -- elements, scan, read -- in values, carry and every gradient, where the passes can go
wrong: lengths around the time tiles and the convolution's width, channel counts around the 256-channel tiles."""
import pytest
import torch

from gpu_util import relerr

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


def _step(cell, x, done, carry, gy, gc, whole):
    leaves = [x, *carry, *cell.parameters()]
    for t in leaves:
        t.grad = None
    if whole:
        out = cell.whole(x, done, carry)
        assert out is not None
        nxt, y = out
    else:
        h, nxt = cell.scan(cell(x), carry, done)
        y = cell.read(h, x)
    loss = (y * gy).sum() + sum((c * g).sum() for c, g in zip(nxt, gc))
    loss.backward()
    return [y, *nxt], [t.grad.clone() for t in leaves]


@pytest.mark.parametrize("B,T,H,P,N,K", [
    (2, 1, 2, 64, 64, 4), (1, 2, 1, 16, 4, 4), (3, 3, 2, 16, 16, 3), (2, 31, 3, 48, 32, 2), (2, 33, 4, 64, 16, 1), (1, 130, 8, 64, 64, 4),
    (5, 65, 5, 52, 64, 4), (70, 34, 2, 32, 32, 4)])
def test_mamba_cell_whole_equals_its_composition(B, T, H, P, N, K):
    from memorax_amd import sequence_models as sm
    torch.manual_seed(T)
    Fe = 24
    cell = sm.MambaCell(Fe, num_heads=H, head_dim=P, state_dim=N, conv_dim=K).cuda()
    g = torch.Generator(device="cuda").manual_seed(B)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x = rand(B, T, Fe).requires_grad_()
    done = torch.rand(B, T, device="cuda", generator=g) < 0.05
    carry = [rand(B, 1, H, N, P).requires_grad_(), torch.rand(B, 1, H, 1, 1, device="cuda", generator=g).requires_grad_()]
    gy, gc = rand(B, T, Fe), [rand(B, 1, H, N, P) * 0.1, rand(B, 1, H, 1, 1)]
    print(f"case mamba {B} {T} {H} {P} {N} {K}", flush=True)
    outs, grads = _step(cell, x, done, carry, gy, gc, True)
    ref_outs, ref_grads = _step(cell, x, done, carry, gy, gc, False)
    names = ["y", "S", "decay"] + ["dx", "dS0", "ddecay0"] + [n for n, _ in cell.named_parameters()]
    for n, a, b in zip(names, outs + grads, ref_outs + ref_grads):
        assert a.shape == b.shape, n
        assert relerr(a, _np(b)) <= 2e-4, (n, relerr(a, _np(b)))


@pytest.mark.parametrize("B,T,H,P,N,K", [(3, 37, 3, 20, 8, 4), (9, 67, 9, 32, 8, 3), (2, 3, 5, 8, 4, 2), (260, 35, 5, 52, 16, 4)])
def test_mamba_cell_narrow_heads_and_tails(B, T, H, P, N, K):
    """Heads narrower than the four lanes that share a step's gates, and tiles that end inside a group of four steps."""
    test_mamba_cell_whole_equals_its_composition(B, T, H, P, N, K)


def test_mamba_cell_acting_equals_its_composition():
    from memorax_amd import sequence_models as sm
    torch.manual_seed(3)
    B, Fe, H, d = 37, 32, 2, 32
    cell = sm.MambaCell(Fe, num_heads=H, head_dim=d, state_dim=d).cuda()
    carry = ref = cell.initialize_carry(None, (B, Fe))
    with torch.no_grad():
        for t in range(4):
            x, done = torch.randn(B, 1, Fe, device="cuda"), torch.rand(B, 1, device="cuda") < 0.2
            carry, y = sm.Memoroid(cell)(x, done, carry)
            h, ref = cell.scan(cell(x), ref, done)
            assert relerr(y, _np(cell.read(h, x))) <= 1e-4
            for a, b in zip(carry, ref):
                assert a.shape == b.shape and relerr(a, _np(b)) <= 1e-4


def test_mamba_cell_notices_a_carry_overwritten_before_the_backward():
    """The decay leaf is read by the backward: a rollout that reuses its buffer in between must not pass in silence."""
    from memorax_amd import sequence_models as sm
    torch.manual_seed(5)
    cell = sm.MambaCell(16, num_heads=2, head_dim=32, state_dim=32).cuda()
    carry = (torch.zeros(3, 1, 2, 32, 32, device="cuda"), torch.full((3, 1, 2, 1, 1), 0.5, device="cuda"))
    nxt, y = cell.whole(torch.randn(3, 5, 16, device="cuda"), torch.zeros(3, 5, dtype=torch.bool, device="cuda"), carry)
    loss = y.sum() + nxt[1].sum()
    carry[1].mul_(2.0)
    with pytest.raises(RuntimeError, match="inplace operation"):
        loss.backward()


@pytest.mark.parametrize("what", ["conv", "mamba"])
def test_saved_tensors_that_a_hook_hands_back_in_another_layout(what):
    """Torch's hooks on saved tensors may hand on copies whose elements lie elsewhere: they are read by their strides."""
    from memorax_amd import _lib, sequence_models as sm
    torch.manual_seed(7)
    if what == "conv":
        x, w, b = torch.randn(3, 9, 16, device="cuda"), torch.randn(16, 1, 4, device="cuda"), torch.randn(16, device="cuda")
        leaves = [t.requires_grad_() for t in (x, w, b)]
        run = lambda: _lib.native().causal_conv_silu(x, w, b)  # noqa: E731
    else:
        cell = sm.MambaCell(16, num_heads=2, head_dim=32, state_dim=32).cuda()
        x, done = torch.randn(3, 9, 16, device="cuda", requires_grad=True), torch.rand(3, 9, device="cuda") < 0.1
        carry = cell.initialize_carry(None, (3, 16))
        leaves = [x, *cell.parameters()]
        run = lambda: cell.whole(x, done, carry)[1]  # noqa: E731
    seen = []

    def unpack(t):
        seen.append(t.dim() > 1)
        return t.transpose(0, -1).contiguous().transpose(0, -1) if t.dim() > 1 else t

    want = torch.autograd.grad(run().square().sum(), leaves)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        loss = run().square().sum()
    got = torch.autograd.grad(loss, leaves)
    assert any(seen)
    for a, b in zip(got, want):   # the same kernels on the same numbers; the projections around Mamba's in another order of their sums
        assert float((a - b).norm()) <= (0.0 if what == "conv" else 1e-5) * float(b.norm())
