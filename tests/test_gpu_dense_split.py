"""Float32 dense layers on the bfloat16 matrix units (csrc/dense_split.hip, the float32 kernels of csrc/dense_grads.hip) against double
precision: sizes around their tiles and steps, rows and columns of very different magnitudes, infinities and NaN."""
import ctypes

import pytest
import torch

from memorax_amd import _lib
from memorax_amd.dense import Weights, dense_group

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _case(rows, K, outs, seed=0):
    g = torch.Generator(device="cuda").manual_seed(rows + K + len(outs) + seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    return rnd(rows, K), [rnd(n, K) for n in outs], [rnd(n) if i % 2 else None for i, n in enumerate(outs)], [rnd(rows, n) for n in outs]


def _run(x, ws, bs, dys):
    x, ws, bs = (t.clone().requires_grad_() if torch.is_tensor(t) else [None if u is None else u.clone().requires_grad_() for u in t] for t in (x, ws, bs))
    ys = dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)])
    torch.autograd.backward(ys, dys)
    for b, dy in zip(bs, dys):   # a sum of rows: sqrt(rows) roundings of a few terms' size, twice over
        if b is not None and bool(torch.isfinite(dy).all()) and dy.dtype == torch.float32:
            d = dy.double()
            assert ((b.grad.double() - d.sum(0)).abs() <= 2 * EPS * (dy.shape[0] * (d ** 2).sum(0)).sqrt() + 1e-38).all()
    return [y.detach() for y in ys], x.grad, [w.grad for w in ws]


def _close(got, a, b, add=None):
    """got = a b (+ add) with a (m, k), b (k, n): an element is out by what splitting leaves of each product (2^-26) and by the roundings of
    its running sum, together within 16 eps of the products' 2-norm -- eight times what they are on average."""
    want = a.double() @ b.double()
    size = (a.double().abs() ** 2 @ b.double().abs() ** 2).sqrt()
    if add is not None:
        want, size = want + add.double(), size + add.double().abs()
    assert ((got.double() - want).abs() <= 16 * EPS * a.shape[1] ** 0.25 * size + 1e-38).all(), float(((got.double() - want).abs() / size.clamp_min(1e-30)).max() / EPS)


@pytest.mark.parametrize("rows,K,outs", [(1, 64, [64, 3]), (63, 64, [1, 16, 17]), (65, 72, [130, 256]), (128, 256, [64, 64, 64, 2]), (129, 264, [48, 260]),
                                         (300, 520, [16, 5, 16]), (4097, 256, [512, 256, 8]), (9000, 128, [128] * 8),
                                         (40000, 64, [64, 8]), (17000, 200, [300, 40])])
def test_sizes(rows, K, outs):
    x, ws, bs, dys = _case(rows, K, outs)
    print(f"case dense split rows={rows} K={K} outs={outs}", flush=True)
    ys, dx, dws = _run(x, ws, bs, dys)
    for y, w, b in zip(ys, ws, bs):
        _close(y, x, w.t(), b)
    _close(dx, torch.cat(dys, 1), torch.cat(ws))
    for dw, dy in zip(dws, dys):
        _close(dw, dy.t(), x)


def test_magnitudes():
    """Rows, columns of the weights and steps of a longer contraction of very different magnitudes."""
    x, ws, bs, dys = _case(500, 520, [300, 16])
    rows, feats = (torch.randint(-40, 40, (n,), generator=torch.Generator().manual_seed(n)).cuda() for n in (500, 300))
    x = torch.ldexp(x, rows[:, None])
    x[:, 256:] = torch.ldexp(x[:, 256:], torch.tensor(-18, device="cuda"))
    x[7], x[8, 256:], x[9, :256] = 0., 0., 0.
    ws[0] = torch.ldexp(ws[0], (feats[:, None] // 4))
    ws[0][3] = 0.
    dys[0][:, :256] = torch.ldexp(dys[0][:, :256], torch.tensor(30, device="cuda"))   # far above what follows it
    ys, dx, dws = _run(x, ws, bs, dys)
    for y, w, b in zip(ys, ws, bs):
        _close(y, x, w.t(), b)
    _close(dx, torch.cat(dys, 1), torch.cat(ws))


@pytest.mark.parametrize("big", [2.0 ** 20, 1e12, 1e18])
def test_outliers_that_meet_zeros(big):
    """A value takes nothing from its row's or column's others, however far above or below them it lies: what the operands hold is in the products,
    also where the large ones meet zeros."""
    x, ws, bs, dys = _case(700, 200, [96, 24])
    x[:, 5], ws[0][:, 5], ws[1][:, 5] = big, 0., 0.                       # a feature that no layer uses
    x[33, 9], ws[0][:, 9], ws[1][:, 9] = -big, 0., 0.
    ws[0][3], ws[0][4], ws[1][2] = ws[0][3] * 2.0 ** -50, ws[0][4] * 1e-28, ws[1][2] * 2.0 ** 41
    ws[0][7, ::2] *= big                                                # a column of wide range
    x[100:164, ::2] = 0.
    x[300:310], x[310:320], x[320:330] = x[300:310] * 2.0 ** -60, x[310:320] * 2.0 ** -90, x[320:330].sign() * (x[320:330].abs() + 1) * 2.0 ** -110
    dys[0][400:420], dys[1][400:420], x[400:420, 7] = 0., 0., big      # rows without gradients
    dys[0][:, 11], ws[0][11] = dys[0][:, 11] * big, 0.
    dys[0][500:600, 12], x[500:600, 13] = big, 0.
    _, dx, dws = _run(x, ws, bs, dys)
    _close(dx, torch.cat(dys, 1), torch.cat(ws))
    for dw, dy in zip(dws, dys):
        _close(dw, dy.t(), x)
    ys, _, _ = _run(x, ws, bs, dys)
    for y, w, b in zip(ys, ws, bs):
        _close(y, x, w.t(), b)


@pytest.mark.parametrize("late", [False, True])
def test_columns_that_grow_along_the_rows(late):
    """The parameters' gradients where a later step of rows goes far beyond the earlier ones, zeros first among them."""
    x, ws, bs, dys = _case(2000, 64, [64, 8])
    x[:, 5], dys[0][:, 9] = 0., 0.
    at = slice(700, None) if late else slice(0, 40)
    x[at, 3] = torch.ldexp(x[at, 3], torch.tensor(30, device="cuda"))
    x[at, 5] = 1e-30
    dys[0][at, 9] = 1e20
    dys[1][at] = torch.ldexp(dys[1][at], torch.tensor(12, device="cuda"))
    _, _, dws = _run(x, ws, bs, dys)
    for dw, dy in zip(dws, dys):
        _close(dw, dy.t(), x)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_what_is_not_finite(bad):
    """What float32 makes of it: infinite or NaN where the operand has a part in the sum, everything else as without it."""
    x, ws, bs, dys = _case(200, 128, [64, 72])
    clean = _run(x, ws, bs, dys)
    x1, w1, dy1 = x.clone(), [w.clone() for w in ws], [d.clone() for d in dys]
    x1[70, 5] = bad
    w1[1][9, 3] = bad
    ys, _, dws = _run(x1, w1, bs, dys)
    for l, y in enumerate(ys):
        want = x1.double() @ w1[l].double().t() + (0 if bs[l] is None else bs[l].double())
        assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isposinf(y), torch.isposinf(want))
        fine = torch.isfinite(want)
        assert (y.double() - want)[fine].abs().max() <= 64 * EPS * 128
    for l, dw in enumerate(dws):
        fine = torch.ones(128, dtype=torch.bool, device="cuda")
        fine[5] = False
        assert not torch.isfinite(dw[:, 5]).any() and (dw - clean[2][l])[:, fine].abs().max() <= 64 * EPS * 200
    dy1[0][70, 9] = bad
    _, dx, dws = _run(x, ws, bs, dy1)
    want = sum(d.double() @ w.double() for d, w in zip(dy1, ws))
    assert torch.equal(torch.isnan(dx), torch.isnan(want)) and torch.equal(torch.isneginf(dx), torch.isneginf(want))
    assert not torch.isfinite(dws[0][9]).any() and torch.isfinite(dws[1]).all() and torch.isfinite(dws[0][:9]).all()


@pytest.mark.parametrize("at", [63, 37, 16])
def test_an_infinity_in_every_tile_of_rows(at):
    """Whichever wave of a workgroup meets it: each tile's row has infinite sums, none of them NaN."""
    x, ws, bs, _ = _case(64 * 700, 64, [64, 64])
    x[at::64, 3] = float("inf")
    ws = [w.requires_grad_() for w in ws]
    for y, w in zip(dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)]), ws):
        assert torch.equal(y[at::64], (w[:, 3].sign() * float("inf")).expand(700, -1))
        assert int(torch.isfinite(y).sum()) == 63 * 700 * 64


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("row", [0, 70, 199])
def test_bias_gradients_of_what_is_not_finite(bad, row):
    """An infinity among the rows is the sum of its column, as in the array library's sums; opposite ones and NaN are NaN."""
    x, ws, _, dys = _case(200, 128, [64, 72])
    dys[0][row, 9], dys[1][row, 3], dys[1][5, 4], dys[1][190, 4] = bad, 1.0, bad, -bad
    bs = [torch.zeros(w.shape[0], device="cuda", requires_grad=True) for w in ws]
    torch.autograd.backward(dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)]), dys)
    for b, dy in zip(bs, dys):
        want = dy.double().sum(0)
        fine = torch.isfinite(want)
        assert torch.equal(torch.isnan(b.grad), torch.isnan(want)) and torch.equal(b.grad.double()[torch.isinf(want)], want[torch.isinf(want)])
        assert (b.grad.double() - want)[fine].abs().max() <= 8 * EPS * 200 ** 0.5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,K,outs", [(64, 131072, [1]), (70, 65544, [3, 1]), (16, 8, [65537, 16]), (300, 8, [131072])])
def test_widths_beyond_the_kernels(rows, K, outs, dtype):
    """More features or outputs than the kernels' 65536: the array library's products, as small as the layers are otherwise."""
    x, ws, _, dys = _case(rows, K, outs)
    x, ws, dys = x.to(dtype), [w.to(dtype) for w in ws], [d.to(dtype) for d in dys]
    print(f"case dense split wide rows={rows} K={K} outs={outs} {dtype}", flush=True)
    _, dx, dws = _run(x, ws, [None] * len(ws), dys)
    if dtype == torch.float32:
        _close(dx, torch.cat(dys, 1), torch.cat(ws))
    else:   # each layer's share, and their sum, is rounded
        want, size = sum(d.double() @ w.double() for d, w in zip(dys, ws)), sum((d.double().abs() @ w.double().abs()) for d, w in zip(dys, ws))
        assert ((dx.double() - want).abs() <= 2.0 ** -7 * size).all()
    for dw, dy in zip(dws, dys):
        if dtype == torch.float32:
            _close(dw, dy.t(), x)
        else:
            want = dy.double().t() @ x.double()
            assert ((dw.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3).all()


def test_bfloat16_input_gradients():
    """An input gradient that is asked for in bfloat16."""
    x, ws, _, dys = _case(1000, 128, [96])
    got = _lib.native().dense_grads(x, dys, ws, [False], True, torch.bfloat16, False)[0]
    want = dys[0].double() @ ws[0].double()
    assert got.dtype == torch.bfloat16 and ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


def _pointers(*ts):
    return (ctypes.c_void_p * len(ts))(*(None if t is None else t.data_ptr() for t in ts))


@pytest.mark.parametrize("bad", [None, float("inf")])
@pytest.mark.parametrize("n", [17, 64])
@pytest.mark.parametrize("rows", [70, 20000])
def test_what_is_added_to_a_layer_s_result(rows, n, bad):
    """The C entries' residual and skip, with and without a bias, in rows of whole 16-byte pieces and others, also where the sums are formed one by one."""
    lib, K = _lib.load(), 72
    x, (w,), _, (dy,) = _case(rows, K, [n])
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    residual, skip, z, b, sx = rnd(rows, n), rnd(n), rnd(rows, n), rnd(n), rnd(K)
    zx = rnd(rows, K)
    if bad is not None:
        x[13, 3], dy[13, 5] = bad, bad
    sizes = (ctypes.c_int64 * 1)(n)
    work = torch.empty(max(lib.mrx_dense_f32_workspace(sizes, 1, K), lib.mrx_dense_f32_input_grad_workspace(sizes, 1, K)), device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    at = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    fine = torch.arange(rows, device="cuda") != (13 if bad is not None else -1)
    for add, sk, bias in [(residual, None, b), (None, skip, None), (residual, skip, b), (None, None, None)]:
        y = torch.full((rows, n), -7.0, device="cuda")
        assert lib.mrx_dense_f32(stream, at(x), _pointers(w), _pointers(bias), _pointers(y), sizes, 1, at(add), at(sk), None if sk is None else at(z), rows, K, at(work)) == 0
        more = sum((t for t in (add, None if sk is None else sk * z, bias) if t is not None), torch.zeros(rows, n, device="cuda"))
        size = more.abs() + (0 if add is None else add.abs()) + (0 if bias is None else bias.abs())
        want = x.double() @ w.double().t() + more.double()
        room = 16 * EPS * (K ** 0.25 * (x.double() ** 2 @ (w.double() ** 2).t()).sqrt() + size)
        assert ((y.double() - want).abs() <= room)[fine].all()
        assert bad is None or torch.equal(y[13].double(), want[13])
    for sk in (None, sx):
        dx = torch.full((rows, K), -7.0, device="cuda")
        assert lib.mrx_dense_f32_input_grad(stream, _pointers(dy), _pointers(w), sizes, 1, at(sk), None if sk is None else at(zx), at(dx), rows, K, at(work)) == 0
        want = dy.double() @ w.double() + (0 if sk is None else (sk * zx).double())
        room = 16 * EPS * (n ** 0.25 * (dy.double() ** 2 @ w.double() ** 2).sqrt() + (0 if sk is None else (sk * zx).abs()))
        assert ((dx.double() - want).abs() <= room)[fine].all()
        assert bad is None or torch.equal(dx[13].double(), want[13])


@pytest.mark.parametrize("rows", [15, 16, 17, 1024, 1025, 2048, 2049, 4096, 4097])
def test_few_rows(rows):
    """Tiles of 16, 32 and 64 rows, and one or two of a workgroup's columns to a wave."""
    for K, outs in ((128, [128, 120, 8]), (256, [256, 40]), (64, [64, 64])):
        x, ws, bs, dys = _case(rows, K, outs)
        print(f"case dense split few rows={rows} K={K} outs={outs}", flush=True)
        ys, dx, dws = _run(x, ws, bs, dys)
        for y, w, b in zip(ys, ws, bs):
            _close(y, x, w.t(), b)
        _close(dx, torch.cat(dys, 1), torch.cat(ws))
        for dw, dy in zip(dws, dys):
            _close(dw, dy.t(), x)


def test_graph_replays():
    """Two launches and no memset: a captured call gives the eager result on every replay."""
    x, ws, bs, dys = _case(700, 128, [64, 64])
    ws = [w.requires_grad_() for w in ws]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ys = dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)])
    for k in range(3):
        x.copy_(torch.randn(x.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(k)))
        want = dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)])
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(ys, want))
