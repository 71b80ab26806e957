"""The acting step of a gated recurrence as one native call (gated_act: gated_step.hip and the closing layer) against the launches it
stands for -- the row kernel, the MinGRU step, the row kernel -- at the edges of its tiles of 16 rows and 64 features and of its weights'
stretch, each pair of types, and where it takes those launches itself."""
import pytest
import torch

from gpu_util import relerr

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def _np(t):
    return t.detach().float().cpu().numpy()


@pytest.mark.parametrize("rows,K,N", [(1, 8, 8), (15, 24, 56), (16, 256, 64), (17, 264, 72), (33, 512, 200), (130, 136, 256),
                                      (5, 520, 64)])   # the last: past its features
@pytest.mark.parametrize("wd,product", [(F32, F32), (F32, BF), (BF, BF)])
@pytest.mark.parametrize("norm,bias", [(0, False), (1, False), (2, False), (1, True)])
def test_gated_act_equals_its_launches(rows, K, N, wd, product, norm, bias):
    from memorax_amd import _lib
    n = _lib.native()
    g = torch.Generator(device="cuda").manual_seed(rows + K + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, scale, nbias = rand(rows, 1, K), rand(K) if norm else None, rand(K) if norm == 2 else None
    ws = [(rand(N, K) * K ** -0.5).to(wd) for _ in range(3)] + [(rand(K, N) * N ** -0.5).to(wd)]
    bs = [rand(w.shape[0]).to(wd) if bias else None for w in ws]
    done = torch.rand(rows, 1, device="cuda", generator=g) < 0.3
    if rows % 2:
        done = done.float()
    ls, ld = rand(rows, 1, N), -torch.rand(rows, 1, N, device="cuda", generator=g)
    ls[0] = -float("inf")   # a carry of zero
    print(f"case gated step {rows} {K} {N} {wd} {product} {norm} {bias}", flush=True)
    u = n.row_dense(x, norm, scale, nbias, 1e-6, False, ws[:3], bs[:3], product, product, None)
    h, want_s, want_d = n.mingru_step(u[0], u[1], u[2], done, ls, ld, False)
    want = n.row_dense(h, 0, None, None, 0.0, False, ws[3:], bs[3:], product, F32, x)[0]
    # the same roundings around sums of up to 520 products in another order: float32's own, or a bfloat16 of z, h~ or gate the other way
    tol = 1e-5 if product == F32 else 2e-2
    for in_place in (False, True):
        a, b = ls.clone(), ld.clone()
        y, z, s, d = n.gated_act(x, norm, scale, nbias, 1e-6, ws, bs, product, done, a, b, in_place)
        assert (s.data_ptr() == a.data_ptr()) == in_place and (d.data_ptr() == b.data_ptr()) == in_place
        assert y.dtype == F32 and z.dtype == product and z.shape == u[0].shape
        assert relerr(y, _np(want)) <= tol and relerr(z, _np(u[0])) <= tol
        assert relerr(s.exp(), _np(want_s.exp())) <= tol and relerr(d, _np(want_d)) <= tol
        if not in_place:
            assert torch.equal(a, ls) and torch.equal(b, ld)
