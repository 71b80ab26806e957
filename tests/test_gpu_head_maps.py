"""Block-diagonal maps of the mLSTM cell (head_maps): values and gradients against float64, on dense rows and on a half of wider
ones, unused outputs, and heads that must not see each other."""
import pytest
import torch

from gpu_util import relerr
from memorax_amd import sequence_models as sm
from memorax_amd._lib import native

pytestmark = pytest.mark.gpu


def _exact(x, m):
    H, o, d = m.shape
    return torch.einsum("...hd,hod->...ho", x.reshape(*x.shape[:-1], H, d), m).reshape(*x.shape[:-1], H * o)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("B,T,H,o,d", [(1, 1, 1, 4, 4), (3, 5, 2, 16, 16), (2, 65, 3, 20, 12), (70, 129, 4, 64, 64), (256, 128, 2, 32, 32), (5, 7, 8, 64, 64),
                                       (40, 257, 1, 64, 36)])
def test_maps_and_gradients(B, T, H, o, d, half):
    g = torch.Generator(device="cuda").manual_seed(B * T)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x = rand(B, T, (1 + half) * H * d).requires_grad_()
    maps = [rand(H, o, d).requires_grad_() for _ in range(3)]
    gs = [rand(B, T, H * o) for _ in range(3)]
    view = x.chunk(2, dim=-1)[0] if half else x
    print(f"case head maps {B} {T} {H} {o} {d} {half}", flush=True)
    ys = native().head_maps(view, maps)
    got = torch.autograd.grad([ys[0], ys[2]], [x, maps[0], maps[2]], [gs[0], gs[2]])   # the second output stays unused
    x64, m64 = x.detach().double().requires_grad_(), [m.detach().double().requires_grad_() for m in maps]
    want = [_exact(x64.chunk(2, dim=-1)[0] if half else x64, m) for m in m64]
    ref = torch.autograd.grad([want[0], want[2]], [x64, m64[0], m64[2]], [gs[0].double(), gs[2].double()])
    for a, b in zip([*ys, *got], [*want, *ref]):
        assert a.shape == b.shape and relerr(a.detach(), b.detach().cpu().numpy()) <= 1e-5
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(native().head_maps(view, maps), ys))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_heads_do_not_see_each_other(bad):
    """A value that is not finite in one head's channels reaches that head's queries, keys, values, gradients and block alone."""
    torch.manual_seed(0)
    B, T, H, d = 4, 40, 4, 32
    cell = sm.mLSTMCell(16, hidden_dim=H * d, num_heads=H).cuda()
    u, g = torch.randn(B, T, H * d, device="cuda"), torch.randn(B, T, H * d, device="cuda")
    u[1, 3, d + 5] = bad
    g[2, 7, 3 * d] = bad
    u.requires_grad_()
    assert cell._maps_native(u)
    q, k = native().head_maps(u, [cell.query.kernel, cell.key.kernel])
    du, dq = torch.autograd.grad([q, k], [u, cell.query.kernel], [g, g])
    for t, head in ((q, 1), (k, 1), (du, 3)):
        finite = torch.isfinite(t.detach()).view(B * T, H, d).all(2).all(0)
        assert finite.tolist() == [h != head for h in range(H)]
    assert torch.isfinite(dq).view(H, -1).all(1).tolist() == [True, False, True, False]


def test_the_cell_keeps_its_heads_apart():
    """The same through the cell's projections: a convolution bias that overflows one head's channel."""
    torch.manual_seed(1)
    cell = sm.mLSTMCell(16, hidden_dim=64, num_heads=4).cuda()
    with torch.no_grad():
        cell.causal_conv.bias[20] = float("inf")
        q, k, v, _, _ = cell._project(torch.randn(2, 9, 16, device="cuda"))
    for t, finite in ((q, [True, False, True, True]), (k, [True, False, True, True]), (v, [True] * 4)):
        assert torch.isfinite(t).all(3).all(1).all(0).tolist() == finite


@pytest.mark.parametrize("i_bias,f_bias", [(False, True), (True, False), (False, False)])
@pytest.mark.parametrize("T", [1, 6])
def test_gates_without_a_bias(i_bias, f_bias, T):
    """A gate whose bias is taken away is a gate with a bias of zero."""
    torch.manual_seed(2)
    block = sm.Residual(sm.PreNorm(sm.Memoroid(sm.mLSTMCell(16, hidden_dim=64, num_heads=2)), 16)).cuda()
    cell = block.module.module.cell
    x, done = torch.randn(3, T, 16, device="cuda"), torch.zeros(3, T, dtype=torch.bool, device="cuda")
    for gate, has in ((cell.i_gate, i_bias), (cell.f_gate, f_bias)):
        if not has:
            gate.bias.data.zero_()
    with torch.no_grad():
        want = block(x, done)[1]
    for gate, has in ((cell.i_gate, i_bias), (cell.f_gate, f_bias)):
        if not has:
            gate.bias = None
    with torch.no_grad():
        y = block(x, done)[1]
    assert relerr(y, want.cpu().numpy()) <= 1e-5
    block(x, done)[1].sum().backward()
    assert all(torch.isfinite(p.grad).all() for p in cell.parameters() if p.grad is not None)
