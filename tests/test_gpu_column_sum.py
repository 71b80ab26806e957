"""The gradient of a broadcast coefficient: its sum over the sequences (mrx_column_sum) at the edges of its 16 groups of rows, four sums each, of
its 64 columns, and on both sides of the number of rows that it takes."""
import pytest
import torch

from memorax_amd import functional as Fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 15, 16, 17, 63, 64, 65, 130, 512, 513])
@pytest.mark.parametrize("D", [1, 33, 64, 65, 184])
@pytest.mark.parametrize("dtype", [torch.float32, torch.complex64, torch.bfloat16])
def test_gradient_of_a_broadcast_coefficient(B, D, dtype):
    print(f"case column sum {B} {D} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B + D)
    E = torch.complex64 if dtype.is_complex else torch.float32
    wide = torch.complex128 if dtype.is_complex else torch.float64
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen, dtype=E)  # noqa: E731
    a, b, g = (rnd(D) * 0.3).to(dtype), rnd(B, 2, D).to(dtype), rnd(B, 2, D).to(dtype)
    done = torch.zeros(B, 2, dtype=torch.bool, device="cuda")
    leaf = a.clone().requires_grad_()
    h = Fn.linear_scan(leaf, b, done)[0]
    (got,) = torch.autograd.grad(h, [leaf], g)
    # two steps, no carry: h_1 = a h_0 + b_1, so da = sum over the sequences of g_1 conj(h_0)
    terms = g[:, 1].to(wide) * b[:, 0].to(wide).conj()
    want = terms.sum(0)
    bound = 2.0 ** -23 * (2 + B // 32 + 6) * terms.abs().sum(0)   # the longest chain of sums, a complex product's two roundings
    if dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * want.abs()
    assert got.dtype == dtype and got.shape == a.shape
    assert ((got.to(wide) - want).abs() <= bound).all()


@pytest.mark.parametrize("rows", [511, 512, 513, 575, 1023, 1025, 4097])
@pytest.mark.parametrize("columns", [1, 15, 16, 17, 256, 4096, 4097])
def test_many_rows(rows, columns):
    """Either side of the rule by which few columns take sixteen per workgroup: 64 threads a column, eight sums each."""
    from memorax_amd import _lib
    print(f"case column sum of many rows {rows} {columns}", flush=True)
    x = torch.randn(rows, columns, device="cuda", generator=torch.Generator(device="cuda").manual_seed(rows + columns))
    out = torch.full((columns + 1,), 7.0, device="cuda")
    assert _lib.load().mrx_column_sum(torch.cuda.current_stream().cuda_stream, x.data_ptr(), out.data_ptr(), rows, columns) == 0
    bound = 2.0 ** -23 * (rows // 64 + 2 + 6) * x.double().abs().sum(0)   # the longest chain of sums, of either kernel
    assert ((out[:-1].double() - x.double().sum(0)).abs() <= bound).all() and out[-1] == 7.0
