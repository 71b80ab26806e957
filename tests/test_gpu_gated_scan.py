"""The gated recurrence in one launch each way (gated_scan: scan.hip with the gate inside), or the scan and the gate apart where that is faster, against the operations
it stands for -- exp of the carry, the MinGRU scan, the gate, the logarithms: the planner's kinds of kernel (wave-split with one, two and four elements a lane, eight and sixteen
waves, eight and sixteen steps; streams; streams that form the states again), ragged widths, short and long sequences, and a carry of zero."""
import pytest
import torch

from gpu_util import relerr

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def _np(t):
    return t.detach().float().cpu().numpy()


# few columns and sixteen waves, eight, four; streams; segments; one step; float32 on four elements a lane, backward on two (300 x 64 x 200, 146 x 113 x 265); streams of two and
# four elements; states formed again (2400 x 64 x 700, 1024 x 128 x 256 float32); apart forward (380 x 240 x 136 bfloat16, 2100 x 45 x 131 float32), backward (280 x 140 x 165
# float32) or both ways (7000 x 30 x 59 and 4700 x 64 x 61 bfloat16)
SHAPES = [(3, 5, 7), (2, 1, 64), (9, 129, 100), (40, 64, 257), (64, 200, 192), (300, 40, 256), (1100, 33, 130), (700, 70, 512), (4, 900, 48), (600, 24, 4), (2400, 64, 700),
          (300, 64, 200), (146, 113, 265), (32, 128, 256), (200, 520, 70), (5894, 21, 120), (3000, 16, 200), (1024, 128, 256), (380, 240, 136), (2100, 45, 131), (7000, 30, 59),
          (280, 140, 165), (4700, 64, 61)]


@pytest.mark.parametrize("B,T,D", SHAPES)
@pytest.mark.parametrize("dt", [F32, BF])
def test_gated_scan_equals_its_operations(B, T, D, dt):
    from memorax_amd import _lib
    from memorax_amd import functional as Fn
    if B * T * D > 1e8 and dt == F32:
        pytest.skip("the largest once")
    g = torch.Generator(device="cuda").manual_seed(B + T + D)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    z, x, gate = (rand(B, T, D).to(dt).requires_grad_() for _ in range(3))
    ls, ld = rand(B, 1, D), -torch.rand(B, 1, D, device="cuda", generator=g)
    ls[0] = -float("inf")   # a state of zero
    ls.requires_grad_()
    done = torch.rand(B, T, device="cuda", generator=g) < 0.1
    if D % 2:
        done = done.float()
    dy, dl = rand(B, T, D).to(dt), rand(B, 1, D)
    print(f"case gated scan {B} {T} {D} {dt}", flush=True)
    y, s, d = _lib.native().gated_scan(z, x, gate, done, ls, ld)
    h, hl, Pl = Fn.mingru_scan(z, x, done, ls.exp()[:, 0], ld.exp()[:, 0])
    want = (Fn.silu_gate(h, gate), hl[:, None].log(), Pl[:, None].log())
    # the same operations in another order of rounding: float32's own, or a bfloat16 of dh more or less
    tol = 1e-5 if dt == F32 else 1e-2
    assert y.dtype == dt and s.shape == d.shape == ls.shape
    assert relerr(y, _np(want[0])) <= tol and relerr(s, _np(want[1])) <= 1e-5
    assert relerr(d.exp(), _np(want[2].exp())) <= 1e-5 and not d.requires_grad
    for outs, ins in (((0,), 3), ((0, 1), 4)):
        grads = [dy, dl]
        got = torch.autograd.grad([(y, s)[i] for i in outs], [z, x, gate, ls][:ins], [grads[i] for i in outs], retain_graph=True)
        ref = torch.autograd.grad([want[i] for i in outs], [z, x, gate, ls][:ins], [grads[i] for i in outs], retain_graph=True)
        for a, b in zip(got, ref):
            assert a.dtype == b.dtype and a.shape == b.shape
            assert relerr(a, _np(b)) <= 2 * tol


def _operations(z, x, gate, done, ls, ld):
    from memorax_amd import functional as Fn
    h, hl, Pl = Fn.mingru_scan(z, x, done, ls.exp()[:, 0], ld.exp()[:, 0])
    return Fn.silu_gate(h, gate), hl[:, None].log(), Pl[:, None].log()


@pytest.mark.parametrize("B,T,D", [(3, 5, 7), (300, 40, 256), (1100, 33, 130)])   # wave-split, and whole rows streaming
def test_carries_overwritten_between_the_passes(B, T, D):
    """A program that keeps its carry in one buffer writes the next one over it, or clears what it was handed, before the backward."""
    from memorax_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(D)
    z, x, gate = (torch.randn(B, T, D, device="cuda", generator=g).requires_grad_() for _ in range(3))
    ls, ld = torch.randn(B, 1, D, device="cuda", generator=g), torch.zeros(B, 1, D, device="cuda")
    done, dy, dl = torch.rand(B, T, device="cuda", generator=g) < 0.1, torch.randn(B, T, D, device="cuda", generator=g), torch.randn(B, 1, D, device="cuda", generator=g)
    want = torch.autograd.grad(_operations(z, x, gate, done, ls.clone(), ld)[:2], (z, x, gate), (dy, dl))
    print(f"case gated scan overwritten {B} {T} {D}", flush=True)
    y, s, d = _lib.native().gated_scan(z, x, gate, done, ls, ld)
    ls.copy_(s.detach())
    ld.copy_(d)
    s.detach().zero_()
    for a, b in zip(torch.autograd.grad((y, s), (z, x, gate), (dy, dl)), want):
        assert relerr(a, _np(b)) <= 2e-5   # as above


def test_gradient_of_the_carry_handed_on():
    """d log h_T / d log h_0 is h_0 / h_T to within a division's and two products' roundings, however far the logarithm is from zero: with every gate shut it is 1."""
    from memorax_amd import _lib
    B, T, D = 40, 3, 96
    ls = torch.rand(B, 1, D, device="cuda") * 160 - 80
    ls.requires_grad_()
    z, x, gate = torch.full((B, T, D), -200.0, device="cuda"), torch.randn(B, T, D, device="cuda"), torch.randn(B, T, D, device="cuda")
    _, s, _ = _lib.native().gated_scan(z, x, gate, torch.zeros(B, T, dtype=torch.bool, device="cuda"), ls, torch.zeros(B, 1, D, device="cuda"))
    (got,) = torch.autograd.grad(s.sum(), ls)
    assert (got - 1).abs().max() <= 3 * 2.0 ** -24


def test_a_carry_of_several_steps_gives_its_first():
    from memorax_amd import _lib
    z, x, gate = (torch.randn(6, 9, 40, device="cuda").requires_grad_() for _ in range(3))
    ls, ld, done = torch.randn(6, 2, 40, device="cuda"), -torch.rand(6, 2, 40, device="cuda"), torch.rand(6, 9, device="cuda") < 0.2
    got, want = _lib.native().gated_scan(z, x, gate, done, ls, ld), _operations(z, x, gate, done, ls, ld)
    for a, b in zip(got, want):
        assert a.shape == b.shape and relerr(a, _np(b)) <= 1e-5


def test_cells_of_their_own_keep_their_scan():
    from memorax_amd import sequence_models as sm
    seen = []

    class Own(sm.MinGRUCell):
        def scan(self, z, carry, done):
            seen.append(1)
            return super().scan(z, carry, done)
    with torch.device("cuda"):
        m = sm.GatedLinearRecurrence(32)
        m.cell = Own(32)
    x, done = torch.randn(2, 5, 32, device="cuda"), torch.zeros(2, 5, dtype=torch.bool, device="cuda")
    m(x, done)
    m.cell = sm.MinGRUCell(32).cuda()
    m.cell.scan = lambda *a: (seen.append(2), sm.MinGRUCell.scan(m.cell, *a))[1]
    m(x, done)
    assert seen == [1, 2]
