"""The gradients of grouped dense layers (mrx_dense_grads) against double precision: widths around the kernels' tiles, layers of a
few outputs whose rows are no whole 16-byte segments, one row to several slices of rows."""
import pytest
import torch

from memorax_amd import _lib

pytestmark = pytest.mark.gpu

CASES = [
    (1, 8, [1]), (63, 64, [3, 64]), (64, 72, [64, 65, 2]), (257, 128, [129, 7, 128, 4]), (1000, 256, [256]),
    (513, 264, [100, 16]), (9001, 64, [8] * 8), (70000, 128, [64, 64, 64, 2]),
]


@pytest.mark.parametrize("rows,K,outs", CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dx_dtype", [torch.float32, torch.bfloat16])
def test_dense_grads(rows, K, outs, dtype, dx_dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + K)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    x, dys, ws = rnd(rows, K), [rnd(rows, n) for n in outs], [rnd(n, K) for n in outs]
    bias = [l % 2 == 0 for l in range(len(outs))]
    print(f"case dense grads rows={rows} K={K} outs={outs} {dtype} {dx_dtype}", flush=True)
    dx, *params = _lib.native().dense_grads(x, dys, ws, bias, True, dx_dtype, True)
    tol = 2e-5

    def check(got, want, t=tol):
        assert (got.double() - want).abs().max() <= t * want.abs().max().clamp_min(1e-30)

    assert dx.dtype == dx_dtype
    check(dx, sum(d.double() @ w.double() for d, w in zip(dys, ws)), 1e-2 if dx_dtype == torch.bfloat16 else tol)
    for l, d in enumerate(dys):
        check(params[l], d.double().t() @ x.double())
        if bias[l]:
            check(params[len(outs) + l], d.double().sum(0))
        else:
            assert params[len(outs) + l] is None or not params[len(outs) + l].numel()
    only = _lib.native().dense_grads(x, dys, ws, bias, False, dx_dtype, True)
    assert all(torch.equal(a, b) for a, b in zip(only[1:], params) if b is not None)


@pytest.mark.parametrize("rows,K,n,biases", [(32768, 256, 256, 0), (32768, 256, 256, 2), (16384, 256, 256, 0), (65536, 128, 256, 1), (65536, 128, 248, 0)])
def test_float32_groups_on_either_side_of_the_rule(rows, K, n, biases):
    """The library's kernels or the array library's slices: float32 sums over the rows, in error against float64 a random walk of
    rounding errors (sqrt(rows) eps of the terms' root mean square), times eight for the longest walk among the elements."""
    import torch
    from memorax_amd.dense import Weights, dense_group
    g = torch.Generator(device="cuda").manual_seed(rows + K + n + biases)
    x = torch.randn(rows, K, device="cuda", generator=g)
    ws = [torch.randn(n, K, device="cuda", generator=g).requires_grad_() for _ in range(3)]
    bs = [torch.randn(n, device="cuda", generator=g).requires_grad_() if i < biases else None for i in range(3)]
    dy = [torch.randn(rows, n, device="cuda", generator=g) for _ in range(3)]
    torch.autograd.backward(dense_group(x, [Weights(w, b) for w, b in zip(ws, bs)]), dy)
    for w, b, d in zip(ws, bs, dy):
        tol = 8 * rows ** 0.5 * 2.0 ** -24 * rows ** 0.5
        assert float((w.grad.double() - d.double().t() @ x.double()).abs().max()) <= tol
        if b is not None:
            assert float((b.grad.double() - d.double().sum(0)).abs().max()) <= tol


@pytest.mark.parametrize("rows,K,outs", [(131072, 256, [256, 256, 256, 4]), (32768, 256, [256, 256, 256, 4]), (1000, 64, [128, 128, 128]), (100, 256, [256, 256])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_sums_keep_float32_s_precision(rows, K, outs, dtype):
    """Rows with a mean, whose sums grow steadily: the parameters' gradients are within 7e-8 of float64 (2-norm; 2^-24 = 6e-8 is one
    rounding of the result, and the partial sums' errors average out over the slices; 1.5e-7 where one slice is all there is, a chain
    of a hundred additions), the input's no further than the array library's products that add up layer by layer."""
    gen = torch.Generator(device="cuda").manual_seed(rows)
    rnd = lambda n: (torch.randn(rows, n, generator=gen, device="cuda") + torch.randn(n, generator=gen, device="cuda")).to(dtype)  # noqa: E731
    x, dys = rnd(K), [rnd(n) for n in outs]
    ws = [(torch.randn(n, K, generator=gen, device="cuda") * K ** -0.5).to(dtype) for n in outs]
    err = lambda got, want: float((got.double() - want).norm() / want.norm())  # noqa: E731
    dx, *params = _lib.native().dense_grads(x, dys, ws, [True] * len(outs), True, torch.float32, True)
    bound = 7e-8 if rows > 100 else 1.6e-7
    for l, d in enumerate(dys):
        assert err(params[l], d.double().t() @ x.double()) <= bound, l
        assert err(params[len(outs) + l], d.double().sum(0)) <= 1.5 * bound, l   # a handful of values: a mean over fewer roundings
    if dtype == torch.float32:
        exact = sum(d.double() @ w.double() for d, w in zip(dys, ws))
        lib = dys[0] @ ws[0]
        for d, w in zip(dys[1:], ws[1:]):
            lib.addmm_(d, w)
        assert err(dx, exact) <= 1.1 * err(lib, exact)


@pytest.mark.parametrize("rows,K,outs,bias", [(98304, 256, [256, 256], True), (98309, 256, [256, 8, 256], True), (65567, 256, [256, 256, 2, 256], False),
                                              (49171, 512, [512], True), (262400, 256, [6, 256, 256, 256], False), (25000, 512, [512, 512], True)])
@pytest.mark.parametrize("shift", [0, 1])
def test_wide_tiles(rows, K, outs, bias, shift):
    """Bfloat16 parameters' gradients on 256 x 256 tiles: rows that end inside a step, one and several rounds, the narrow layer in every
    place, and (shift) a gradient off the boundaries of whole requests, which takes the other kernel.  Bounds as above."""
    gen = torch.Generator(device="cuda").manual_seed(rows)
    print(f"case wide tiles rows={rows} K={K} outs={outs} bias={bias} shift={shift}", flush=True)
    rnd = lambda n: (torch.randn(rows, n, generator=gen, device="cuda") + torch.randn(n, generator=gen, device="cuda")).to(torch.bfloat16)  # noqa: E731
    x, dys = rnd(K), [rnd(n) for n in outs]
    if shift:
        at = next(l for l, n in enumerate(outs) if n > 8)
        flat = torch.empty(dys[at].numel() + 4, device="cuda", dtype=torch.bfloat16)
        flat[4:] = dys[at].flatten()
        dys[at] = flat[4:].view(rows, -1)
    _, *params = _lib.native().dense_grads(x, dys, [], [bias] * len(outs), False, torch.bfloat16, True)
    err = lambda got, want: float((got.double() - want).norm() / want.norm())  # noqa: E731
    for l, d in enumerate(dys):
        assert err(params[l], d.double().t() @ x.double()) <= 7e-8, l
        if bias:
            assert err(params[len(outs) + l], d.double().sum(0)) <= 1.05e-7, l
