"""Dense layers whose weights wait in registers (mrx_dense_rows, mrx_dense_rows_input_grad) against double precision: rows around the
tiles and the ring of tiles, each width and number of layers, the narrow layer, the closing layer of a residual branch."""
import ctypes

import pytest
import torch

from memorax_amd import _lib

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
ROWS = [1, 15, 33, 64, 700, 20011]


def _ptrs(ts):
    return (ctypes.c_void_p * 8)(*[None if t is None else t.data_ptr() for t in ts])


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _rounded(got, exact, terms, eps=2.0 ** -8):
    """One rounding of the result (eps: bfloat16's half unit and a margin of two) and the float32 sums' own (2^-24 of the terms' sum
    of magnitudes an addition)."""
    assert ((got.double() - exact).abs() <= eps * exact.abs() + terms).all()


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("K,outs,bias", [(64, [64], True), (64, [72, 72, 72, 2], False), (128, [128, 128, 128, 4], True), (128, [256, 256], False),
                                         (256, [256, 256, 256, 3], True), (256, [64, 64, 64, 8], False), (256, [1000], True)])
def test_forward_and_input_gradient(rows, K, outs, bias):
    lib = _lib.load()
    print(f"case dense rows {rows} {K} {outs} {bias}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    n = (ctypes.c_int64 * 8)(*outs)
    suit = lib.mrx_dense_rows_suit(rows, K, n, len(outs))
    assert suit & 1
    x, params = rnd(rows, K).to(BF), [rnd(o, K) * K ** -0.5 for o in outs]
    bs = [rnd(o) if bias else None for o in outs]
    ws = [torch.empty_like(w, dtype=BF) for w in params]
    wide = sum(o for o in outs if o > 8)
    wt = torch.empty(K, wide, device="cuda", dtype=BF)
    assert lib.mrx_dense_pack(_stream(), _ptrs(params), n, len(outs), K, _lib.MRX_F32, _ptrs(ws), wt.data_ptr()) == 0
    assert all(torch.equal(w, p.to(BF)) for w, p in zip(ws, params))
    assert torch.equal(wt, torch.cat([w.t() for w, o in zip(ws, outs) if o > 8], 1))
    ys = [torch.full((rows + 3, o), 7.0, device="cuda", dtype=BF) for o in outs]   # rows past the last stay as they are
    assert lib.mrx_dense_rows(_stream(), x.data_ptr(), _ptrs(ws), _ptrs(bs), _ptrs(ys), n, len(outs), None, rows, K, _lib.MRX_F32) == 0
    for y, w, b in zip(ys, ws, bs):
        b16 = 0.0 if b is None else b.to(BF).double()
        _rounded(y[:rows], x.double() @ w.double().t() + b16, (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + abs(b16)))
        assert (y[rows:] == 7.0).all()
    if not suit & 4:
        assert lib.mrx_dense_rows_input_grad(_stream(), _ptrs(ys), n, len(outs), wt.data_ptr(), None, ys[0].data_ptr(), None, rows, K, _lib.MRX_BF16) == -2
        return
    dys = [rnd(rows, o).to(BF) for o in outs]
    dx = torch.full((rows + 3, K), 7.0, device="cuda", dtype=BF)
    narrow = next((w.data_ptr() for w, o in zip(ws, outs) if o <= 8), None)
    assert lib.mrx_dense_rows_input_grad(_stream(), _ptrs(dys), n, len(outs), wt.data_ptr(), narrow, dx.data_ptr(), None, rows, K, _lib.MRX_BF16) == 0
    _rounded(dx[:rows], sum(d.double() @ w.double() for d, w in zip(dys, ws)),
             sum(outs) * 2.0 ** -24 * sum(d.double().abs() @ w.double().abs() for d, w in zip(dys, ws)))
    assert (dx[rows:] == 7.0).all()


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("n", [64, 128, 256])
def test_the_layer_that_closes_a_residual_branch(rows, K, n):
    lib = _lib.load()
    print(f"case closing layer {rows} {K} {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows + K + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, w, b, res = rnd(rows, K).to(BF), (rnd(n, K) * K ** -0.5).to(BF), rnd(n).to(BF), rnd(rows, n)
    ns = (ctypes.c_int64 * 8)(n)
    y = torch.full((rows + 3, n), 7.0, device="cuda")
    assert lib.mrx_dense_rows(_stream(), x.data_ptr(), _ptrs([w]), _ptrs([b]), _ptrs([y]), ns, 1, res.data_ptr(), rows, K, _lib.MRX_BF16) == 0
    terms = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs() + res.double().abs())
    branch = x.double() @ w.double().t() + b.double()
    _rounded(y[:rows], res.double() + branch, terms + 2.0 ** -8 * branch.abs(), 2.0 ** -23)   # (the branch's result is bfloat16)
    assert (y[rows:] == 7.0).all()
    # backward: the stream's gradient is float32, its rounded copy what the products read
    dy, wt = rnd(rows, n), w.t().contiguous()
    dx, copy = torch.full((rows + 3, K), 7.0, device="cuda", dtype=BF), torch.full((rows + 3, n), 7.0, device="cuda", dtype=BF)
    assert lib.mrx_dense_rows_input_grad(_stream(), _ptrs([dy]), ns, 1, wt.data_ptr(), None, dx.data_ptr(), copy.data_ptr(), rows, K, _lib.MRX_F32) == 0
    assert torch.equal(copy[:rows], dy.to(BF)) and (copy[rows:] == 7.0).all() and (dx[rows:] == 7.0).all()
    d = dy.to(BF).double()
    _rounded(dx[:rows], d @ w.double(), n * 2.0 ** -24 * (d.abs() @ w.double().abs()))


def _rows_past_the_counted_wait():
    """A workgroup's first tiles wait for its requests alone; from the tile on that reuses the ring's first place (the eighth of at most 64
    rows) its stores are counted among them.  Every workgroup -- one a compute unit -- gets so far, some of them two tiles farther."""
    return 64 * 8 * torch.cuda.get_device_properties(0).multi_processor_count + 64 * 300 + 37


@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("n", [64, 128, 256])
@pytest.mark.parametrize("wide,narrow", [(1, 0), (2, 0), (3, 0), (3, 4)])
def test_every_forward_and_input_gradient_past_the_counted_wait(K, n, wide, narrow):
    test_forward_and_input_gradient(_rows_past_the_counted_wait(), K, [n] * wide + [narrow] * (narrow > 0), True)


@pytest.mark.parametrize("K", [64, 128, 256])
@pytest.mark.parametrize("n", [64, 128, 256])
def test_every_closing_layer_past_the_counted_wait(K, n):
    test_the_layer_that_closes_a_residual_branch(_rows_past_the_counted_wait(), K, n)


def _block(kind, F, H, d):
    from memorax_amd import sequence_models as sm
    model = {"delta": lambda: sm.Memoroid(sm.DeltaNetCell(F, d, H)), "attention": lambda: sm.Memoroid(sm.LinearAttentionCell(F, d, H)),
             "recurrence": lambda: sm.GatedLinearRecurrence(F)}[kind]()
    return sm.Residual(sm.PreNorm(model, F, norm=sm.RMSNorm)).cuda()


@pytest.mark.parametrize("kind", ["delta", "attention", "recurrence"])
@pytest.mark.parametrize("B,T,F,H,d", [(3, 7, 64, 2, 32), (5, 40, 128, 2, 64), (2, 33, 256, 4, 64), (2, 20, 96, 2, 16)])
def test_residual_blocks_close_with_their_sum(kind, B, T, F, H, d):
    """The block with its last layer and the residual sum as one operation, against the composition (which a hook brings back): another
    order of the products' sums, which bfloat16 rounds 2^-8 apart, in the result and in each gradient; 96 features take the composition."""
    torch.manual_seed(F)
    print(f"case block {kind} {B} {T} {F}", flush=True)
    block = _block(kind, F, H, d)
    x, done, gy = torch.randn(B, T, F, device="cuda"), torch.rand(B, T, device="cuda") < 0.05, torch.randn(B, T, F, device="cuda")

    def run():
        xs = x.clone().requires_grad_()
        block.zero_grad()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            carry, y = block(xs, done, block.initialize_carry(None, (B, F)))
        name = type(y.grad_fn).__name__
        y.backward(gy)
        return name, [y.detach(), xs.grad, *[p.grad.clone() for p in block.parameters()], *carry]

    name, got = run()
    handle = block.module.module.register_forward_hook(lambda *a: None)
    plain, want = run()
    handle.remove()
    assert plain != name or F == 96
    assert got[0].dtype == torch.float32
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and float((a.float() - b.float()).detach().norm()) <= 2e-2 * float(b.detach().float().norm())
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        _, y = block(x, done, block.initialize_carry(None, (B, F)))
    assert float((y - got[0]).norm()) <= 1e-2 * float(got[0].norm())


def test_the_sum_falls_back_to_the_array_library():
    n = _lib.native()
    x, w, b, res = torch.randn(4, 5, 64, device="cuda"), torch.randn(64, 64, device="cuda"), torch.randn(64, device="cuda"), torch.randn(4, 5, 64, device="cuda")
    want = res + torch.nn.functional.linear(x, w, b)
    torch.testing.assert_close(n.dense_onto(res, x, w, b), want)                                # float32 products
    torch.testing.assert_close(n.dense_onto(res[:1], x, w, b), res[:1] + torch.nn.functional.linear(x, w, b))   # a sum that broadcasts
    torch.testing.assert_close(n.dense_onto(res.transpose(0, 1).contiguous().transpose(0, 1), x, w, b), want)
    half = n.dense_onto(res.to(BF), x.to(BF), w.to(BF), b.to(BF))
    assert half.dtype == BF
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(res.to(BF).float(), torch.ones_like(res))
        out = n.dense_onto(dual, x.to(BF), w.to(BF), b.to(BF))
        assert torch.equal(torch.autograd.forward_ad.unpack_dual(out).tangent, torch.ones_like(res))


@pytest.mark.parametrize("onto", [False, True])
@pytest.mark.parametrize("unpacked", ["as saved", "another layout"])
def test_hooks_on_saved_tensors_see_the_transposed_weights(onto, unpacked):
    """Everything the node keeps for its backward passes torch's hooks (offloading, checkpoints); what they hand back in another layout is
    read as it is."""
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    w, b, x0, res, gy = (rnd(64, 128) / 11).requires_grad_(), rnd(64).requires_grad_(), rnd(700, 128).to(BF), rnd(700, 64), rnd(700, 64)
    shapes = []

    def run(hooks):
        x = x0.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF), hooks:
            y = _lib.native().dense_onto(res, x, w, b) if onto else _lib.native().dense_group(x, [w], [b])[0]
        return torch.autograd.grad(y, [x, w, b], gy.to(y.dtype))

    def pack(t):
        shapes.append(tuple(t.shape))
        return t.cpu()

    def unpack(t):
        t = t.cuda()
        return t if unpacked == "as saved" else t.t().contiguous().t()

    want, got = run(torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t)), run(torch.autograd.graph.saved_tensors_hooks(pack, unpack))
    assert sorted(shapes) == [(64, 128), (128, 64), (700, 128)]   # the weights, the same transposed, the rows
    for a, b in zip(got, want):   # the same kernels, or the array library's sums of 64 and 700 products in another order, rounded to bfloat16
        assert torch.equal(a, b) if unpacked == "as saved" else float((a - b).norm()) <= 2.0 ** -7 * float(b.norm())
