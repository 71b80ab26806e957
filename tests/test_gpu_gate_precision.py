"""silu and sigmoid in the fused cells to float32's last bits over the range where they are small: |error| <= 4e-7 of each value.
The bound: the exponential 1 ulp (1.2e-7), and half an ulp (6e-8) each for 1 + e, the quotient and the products with exact factors
(at most two).  An exponential that errs in proportion to its argument is off by up to 8e-7 at -14."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BOUND = 4e-7
RANGE = (-14.0, 6.0)


def _values(n):
    return torch.linspace(*RANGE, n, device="cuda")


def _check(got, want):
    worst = ((got.double() - want).abs() / want.abs().clamp_min(1e-30)).max()
    assert float(worst) <= BOUND, float(worst)


@pytest.mark.parametrize("C", [64, 260])
def test_silu_behind_the_convolution_and_its_gradient(C):
    from memorax_amd._lib import native
    s = _values(40 * C).view(1, 40, C)
    x = s.clone().requires_grad_()
    y = native().causal_conv_silu(x, torch.ones(C, 1, 1, device="cuda"), torch.zeros(C, device="cuda"))   # one tap of one: s itself
    ref = s.double().requires_grad_()
    want = torch.nn.functional.silu(ref)
    _check(y.detach(), want.detach())
    (gx,) = torch.autograd.grad(y.sum(), x)
    (gr,) = torch.autograd.grad(want.sum(), ref)
    # sigma (1 + s (1 - sigma)): the sum cancels near its zero at -1.28, where its own rounding (a few 6e-8 of its terms) counts
    sigma = torch.sigmoid(ref.detach())
    assert float(((gx.double() - gr).abs() / (sigma * (1 + ref.detach().abs() * (1 - sigma)))).max()) <= 1.5 * BOUND


@pytest.mark.parametrize("H,D", [(4, 16), (1, 64), (4, 64)])
def test_silu_in_the_mlstm_step(H, D):
    """Read through a skip of one, a norm weight that drops the recurrence and a gate whose silu is exact (30)."""
    from memorax_amd._lib import native
    W = H * D
    dev = dict(device="cuda")
    s = _values(W)
    zeros, eye = torch.zeros(H, D, D, **dev), torch.eye(W, **dev)
    up = torch.cat([torch.zeros(W, W, **dev), 30e20 * eye])
    gates = [torch.zeros(H, 3 * W, **dev), torch.zeros(H, **dev)] * 2
    params = [up, torch.zeros(W, 1, 4, **dev), s, zeros, zeros, zeros, *gates, torch.full((H, D), -1.0, **dev), torch.ones(W, **dev), eye]
    carry = [torch.zeros(2, 1, H, D, D, **dev), torch.zeros(2, 1, H, 1, 1, **dev), torch.zeros(2, 1, H, D, 1, **dev), torch.zeros(2, 1, H, 1, 1, **dev)]
    x = torch.full((2, 1, W), 1e-20, **dev)
    y = native().mlstm_act(x, 0, None, None, 0.0, params, torch.zeros(2, 1, **dev), carry, -60.0)[0]
    scale = x.double()[0, 0] * up.double()[W:].diagonal()
    _check(y[0, 0], torch.nn.functional.silu(s.double()) * scale)


def test_sigmoid_and_key_norm_in_the_delta_rule_step():
    """From an empty state o = sigmoid(beta) v (k . q) / |k|: with k along one axis of a value that norm and quotient keep exact."""
    from memorax_amd._lib import native
    B, H, d = 256, 8, 64
    k = torch.zeros(B, 1, H, d, device="cuda")
    k[..., 3] = 2.0
    q = torch.zeros_like(k)
    q[..., 3] = 1.0
    beta = _values(B * H).view(B, 1, H)
    o, _ = native().delta_rule(q, k, torch.ones_like(k), beta, torch.zeros(B, 1, device="cuda"), None, True, 0, False)
    _check(o, torch.sigmoid(beta.double())[..., None].expand(B, 1, H, d))
