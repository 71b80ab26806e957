"""The residual sum of a float32 stream and a bfloat16 branch (mrx_residual_add): the array library's numbers and derivatives, bit for
bit, at sizes around a thread's eight elements, a workgroup's and the largest grid, and on the arrays it hands back."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2048, 2049, 690_688, 8192 * 2048 + 13])
def test_sum_and_gradients(n):
    from memorax_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, device="cuda", generator=g)
    b = torch.randn(n, device="cuda", generator=g).to(torch.bfloat16)
    x[0], b[-1] = float("inf"), float("nan")
    gy = torch.randn(n, device="cuda", generator=g)
    a = [t.clone().requires_grad_() for t in (x, b)]
    c = [t.clone().requires_grad_() for t in (x, b)]
    one, two = _lib.native().residual_add(*a), c[0] + c[1]
    assert one.dtype == torch.float32 and torch.equal(one.view(torch.int32), two.view(torch.int32))
    for s, t in zip(torch.autograd.grad(one, a, gy), torch.autograd.grad(two, c, gy)):
        assert s.dtype == t.dtype and torch.equal(s, t)


def test_what_the_kernel_does_not_take_and_second_derivatives():
    from memorax_amd import _lib
    add = _lib.native().residual_add
    x, b = torch.randn(6, 4, 8, device="cuda"), torch.randn(6, 4, 8, device="cuda").to(torch.bfloat16)
    for p, q in ((x.transpose(0, 1), b.transpose(0, 1)), (x, b[:1]), (x.flatten()[1:9], b.flatten()[1:9]), (x[:0], b[:0]), (x, b.float())):
        assert torch.equal(add(p, q), p + q)
    with torch.autograd.forward_ad.dual_level():
        t = torch.autograd.forward_ad.unpack_dual(add(torch.autograd.forward_ad.make_dual(x, x), b)).tangent
        assert torch.equal(t, x)
    p, q = x.clone().requires_grad_(), b.clone().requires_grad_()
    (first,) = torch.autograd.grad((add(p, q) ** 3).sum(), p, create_graph=True)
    (second,) = torch.autograd.grad(first.sum(), q)
    want = 6 * (x + b)
    assert torch.allclose(second.float(), want, rtol=2 ** -7, atol=0)   # bfloat16's rounding of the gradient
