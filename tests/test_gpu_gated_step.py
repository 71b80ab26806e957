"""The acting step of a gated recurrence as one native call (gated_act: act_chain.hip and the closing layer) against the launches it
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
                                      (4112, 72, 64), (1040, 128, 256), (1040, 512, 264),   # more workgroups than compute units, two on each and one
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


def _exact_step(x, norm, scale, nbias, eps, ws, bs, product, done, ls, ld):
    """The step in float64 on the weights as the products read them, and how far each result may be from it: products of K rounded operands
    (their roundings independent of each other: six standard deviations of their sum), float32 sums (K + 8 roundings of the terms'
    magnitudes), one rounding of z, h~, gate, the state, the gated state and the closing layer's result each, carried through the maps
    by their slopes (sigma 1/4, g 1, silu 1.1, log sigma 1); 2^-21 of a value for each of the elementary functions."""
    d = lambda t: None if t is None else t.double()  # noqa: E731
    u, f = (2.0 ** -8 if product == BF else 2.0 ** -24), 2.0 ** -24
    ws, bs = [w.to(product).double() for w in ws], [d(b) for b in bs]
    xd = x.double()[:, 0]
    K, N = xd.shape[1], ws[0].shape[0]
    c = xd - xd.mean(-1, keepdim=True) if norm == 2 else xd
    rstd = torch.rsqrt((c * c).mean(-1, keepdim=True) + eps) if norm else torch.ones_like(xd[:, :1])
    s = d(scale) if norm else 1.0
    xn = c * rstd * s + (d(nbias) if nbias is not None else 0.0)
    off = (K + 8) * f * (rstd * abs(s) * (xd.abs() + xd.abs().mean(-1, keepdim=True)) + (nbias.double().abs() if nbias is not None else 0.0)) if norm else 0.0

    def layer(rows, rows_off, w, b):
        y = rows @ w.t() + (0.0 if b is None else b)
        terms = rows.abs() @ w.abs().t() + (0.0 if b is None else b.abs())
        e = (w.shape[1] + 8) * f * terms + 6 * 3 ** -0.5 * u * ((rows * rows) @ (w * w).t()).sqrt() + u * y.abs()
        return y, e + (0.0 if isinstance(rows_off, float) else rows_off @ w.abs().t()) + (0.0 if b is None else u * b.abs())

    (z, ez), (xh, ex), (gate, eg) = (layer(xn, off, w, b) for w, b in zip(ws[:3], bs[:3]))
    g = torch.where(xh >= 0, xh + 0.5, torch.sigmoid(xh))
    a, sg = torch.sigmoid(-z), torch.sigmoid(z)
    b, eb = sg * g, g * ez / 4 + sg * ex + 2.0 ** -21 * sg * g
    reset, carry = done != 0, ls.double()[:, 0].exp()
    h = torch.where(reset, b, a * carry + b)
    eh = torch.where(reset, eb, eb + carry * (ez / 4 + 2.0 ** -21 * a)) + f * h
    log_a = torch.nn.functional.logsigmoid(-z)
    decay = torch.where(reset, log_a, ld.double()[:, 0] + log_a)
    hid, ehid = h * torch.nn.functional.silu(gate), (eh + u * h) * torch.nn.functional.silu(gate).abs() + h * 1.1 * eg
    ehid = ehid + (u + 2.0 ** -21) * hid.abs()
    y, ey = layer(hid, 0.0, ws[3], bs[3])
    ey = ey + 6 * ((ehid * ehid) @ (ws[3] * ws[3]).t()).sqrt()
    return {"y": (y + xd, ey + f * (y + xd).abs()), "z": (z, ez), "state": (h, eh + 2.0 ** -21 * (1 + h.log().abs()) * h),
            "decay": (decay, ez + 2.0 ** -21 * (decay.abs() + log_a.abs()))}


@pytest.mark.parametrize("rows,K,N", [(1, 8, 8), (15, 24, 56), (16, 256, 64), (17, 264, 72), (33, 512, 200), (130, 136, 256), (1024, 256, 256)])
@pytest.mark.parametrize("wd,product", [(F32, F32), (F32, BF), (BF, BF)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_gated_act_against_float64(rows, K, N, wd, product, norm):
    from memorax_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows + K + N + norm)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, scale, nbias = rand(rows, 1, K), rand(K) if norm else None, rand(K) if norm == 2 else None
    ws = [(rand(N, K) * K ** -0.5).to(wd) for _ in range(3)] + [(rand(K, N) * N ** -0.5).to(wd)]
    done = torch.rand(rows, 1, device="cuda", generator=g) < 0.3
    ls, ld = rand(rows, 1, N), -torch.rand(rows, 1, N, device="cuda", generator=g)
    ls[0] = -float("inf")   # a carry of zero
    print(f"case gated step float64 {rows} {K} {N} {wd} {product} {norm}", flush=True)
    y, z, s, decay = _lib.native().gated_act(x, norm, scale, nbias, 1e-6, ws, [None] * 4, product, done, ls, ld, False)
    got = {"y": y, "z": z, "state": s.double().exp(), "decay": decay}
    for name, (want, bound) in _exact_step(x, norm, scale, nbias, 1e-6, ws, [None] * 4, product, done, ls, ld).items():
        err = (got[name].double()[:, 0] - want).abs()
        print(name, float((err / bound).max()), float(err.norm() / want.norm()))
        assert (err <= bound).all(), (name, float((err / bound).max()))
