"""The normalised and the gated form cut along time (a workgroup per chunk, functional's choice on few sequences) against the
sequential pair of kernels.py: values, carries and every gradient, from the smallest number of chunks the rule takes to a ragged
end, whole and narrow heads, few and many resets, with and without carries.

Both are measured against the masked products over the whole sequence in float64 on the same (rounded) inputs.  No result's error is
larger than the sequential pair's: over all cases below the mean ratio is 0.4 to 1.01, and 1.02 at most for any one, but for the
three results that the two splits sum in another order (dg, z, dz0: means of 0.6 to 1.01, single cases up to 1.35, two roundings
of one size).  1e-7 on top is float32's own rounding of a result, for where the other happens to be exact."""
import pytest
import torch

from memorax_amd import functional as Fn
from memorax_amd import kernels as K

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 64, 64, 8.0), (2, 2, 64, 48, 8.4), (3, 1, 32, 32, 10.02), (2, 4, 16, 32, 14.5), (1, 3, 48, 64, 17.0), (16, 8, 32, 32, 10.0)]
TYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _inputs(shape, dtype, p, carries, seed):
    B, H, dk, dv, chunks = shape
    T = round(chunks * (64 if dtype == "bf16" else 32))
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    q, k, v, do = (rnd(B, T, H, d).mul(0.125).to(TYPES[dtype]) for d in (dk, dk, dv, dv))
    gate = -0.1 * torch.rand(B, T, H, device="cuda", generator=g)
    done = torch.rand(B, T, device="cuda", generator=g) < p
    S0, z0, dS, dz = rnd(B, H, dv, dk) * 0.1, torch.rand(B, H, dk, device="cuda", generator=g), rnd(B, H, dv, dk), rnd(B, H, dk)
    dss = rnd(B, T, H)
    if not carries:
        S0 = z0 = None
    assert K.linear_attn_chunk_parallel_pays(B, T, H, TYPES[dtype])
    return q, k, v, gate, do, done, S0, z0, dS, dz, dss


def _distance(a, b):
    return float((a.detach().double() - b).norm() / b.norm().clamp_min(1e-30))


def _compare(got, own, yard):
    for name in yard:
        far, near = _distance(got[name], yard[name]), _distance(own[name], yard[name])
        assert far <= (1.5 if name in ("dg", "z", "dz0") else 1.05) * near + 1e-7, (name, far, near)


def _exact(q, k, v, gate, done, S0, z0, fmap, normalise):
    """(o, S_last) or (o, S_last, z_last, ss) in float64; gate None: no decay."""
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))   # (B,H,T,d)
    if fmap == "elu1":
        q, k = torch.nn.functional.elu(q) + 1, torch.nn.functional.elu(k) + 1
    T = q.shape[2]
    episode = done.cumsum(1)
    pair = (episode[:, :, None] == episode[:, None, :]) & torch.ones(T, T, dtype=torch.bool, device=q.device).tril()
    G = torch.zeros_like(q[..., 0]) if gate is None else gate.transpose(1, 2).cumsum(-1)
    first, last = (episode == 0)[:, None, :], (episode == episode[:, -1:])[:, None, :]
    zero = torch.zeros((), dtype=torch.float64, device=q.device)
    decay = torch.where(pair[:, None], torch.exp(torch.where(pair[:, None], G[..., :, None] - G[..., None, :], zero)), zero)
    A = (q @ k.transpose(-1, -2)) * decay
    a0 = torch.where(first, G.exp(), zero)[..., None]    # what the carried state is worth in each step
    b = torch.where(last, torch.exp(torch.where(last, G[..., -1:] - G, zero)), zero)[..., None]
    o, S = A @ v, (v * b).transpose(-1, -2) @ k
    if S0 is not None:
        o, S = o + a0 * (q @ S0.transpose(-1, -2)), S + a0[..., -1:, :] * S0
    if not normalise:
        return o.transpose(1, 2), S
    den, z = A.sum(-1, keepdim=True), (k * b).sum(2)
    if z0 is not None:
        den, z = den + a0 * (q * z0[:, :, None]).sum(-1, keepdim=True), z + a0[..., -1, :] * z0
    o = o / den.clamp_min(1e-6)
    return o.transpose(1, 2), S, z, o.square().sum(-1).transpose(1, 2)


def _exact_with_gradients(leaves, done, fmap, normalise, cotangents):
    """leaves: q, k, v, gate, S0, z0 (the last three perhaps None)."""
    x = [None if t is None else t.detach().double().requires_grad_() for t in leaves]
    out = _exact(*x[:4], done, *x[4:], fmap, normalise)[:len(cotangents)]
    grads = torch.autograd.grad(out, [t for t in x if t is not None], [t.double() for t in cotangents])
    return [t.detach() for t in out], list(grads)


@pytest.mark.parametrize("carries", [False, True])
@pytest.mark.parametrize("p", [0.0, 0.01, 0.3])
@pytest.mark.parametrize("fmap", ["none", "elu1"])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_gated(shape, dtype, fmap, p, carries):
    q, k, v, gate, do, done, S0, _, dS, _, _ = _inputs(shape, dtype, p, carries, 3)
    fm = int(fmap == "elu1")

    o, S, chk = K.gated_linear_attn_fwd(q, k, v, gate, done, S0, fm)
    names = ["o", "S", "dq", "dk", "dv", "dg"] + ["dS0"] * carries
    own = dict(zip(names, (o, S, *K.gated_linear_attn_bwd(q, k, v, gate, done, chk, do, dS, fm, True, S))))
    out, grads = _exact_with_gradients((q, k, v, gate, S0, None), done, fmap, False, (do, dS))
    yard = dict(zip(names, out + grads))
    leaves = [t.requires_grad_() for t in (q, k, v, gate)] + ([S0.requires_grad_()] if carries else [])
    o, S = Fn.gated_linear_attention(q, k, v, gate, done, S0, fmap)
    got = dict(zip(names, (o, S, *torch.autograd.grad((o, S), leaves, (do, dS)))))
    with torch.no_grad():
        o2, S2 = Fn.gated_linear_attention(q, k, v, gate, done, S0, fmap)
    assert torch.equal(o, o2) and torch.equal(S, S2)
    _compare(got, own, yard)


@pytest.mark.parametrize("carries", [False, True])
@pytest.mark.parametrize("p", [0.0, 0.01, 0.3])
@pytest.mark.parametrize("ss", [False, True])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_normalised(shape, dtype, ss, p, carries):
    q, k, v, _, do, done, S0, z0, dS, dz, dss = _inputs(shape, dtype, p, carries, 5)

    o, den, S, z, chk, *rest = K.linear_attn_norm_fwd(q, k, v, done, S0, z0, 1, 1e-6, True, ss)
    names = ["o", "S", "z"] + ["ss"] * ss + ["dq", "dk", "dv"] + ["dS0", "dz0"] * carries
    own = dict(zip(names, (o, S, z, *rest, *K.linear_attn_norm_bwd(q, k, v, done, chk, o, den, do, dS, dz, 1, 1e-6, True,
                                                                   dss.transpose(1, 2).contiguous() if ss else None))))
    if ss:
        own["ss"] = own["ss"].transpose(1, 2)
    cotangents = (do, dS, dz) + ((dss,) if ss else ())
    out, grads = _exact_with_gradients((q, k, v, None, S0, z0), done, "elu1", True, cotangents)
    yard = dict(zip(names, out + grads))
    leaves = [t.requires_grad_() for t in (q, k, v)] + ([S0.requires_grad_(), z0.requires_grad_()] if carries else [])
    out = Fn.normalised_linear_attention(q, k, v, done, S0, z0, "elu1", return_ss=ss)
    got = dict(zip(names, (*out, *torch.autograd.grad(out, leaves, cotangents))))
    _compare(got, own, yard)


LONG = [(2, 1, 32, 64, 16.0), (1, 2, 64, 64, 31.6), (1, 1, 48, 32, 33.0), (2, 1, 64, 64, 64.0), (1, 2, 32, 32, 65.1), (1, 1, 64, 48, 129.4),
        (16, 8, 64, 64, 16.5)]


@pytest.mark.parametrize("p", [0.0, 0.002])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shape", LONG)
def test_long_scans_of_the_state(shape, dtype, p):
    """As many chunks as slots are on their way (32, and 8 where there are many sequences) or share their flags (64), and a few more.  A slot
    or a flag of the wrong chunk errs by the size of the result; bfloat16 operands of up to three products in a row (2^-9 each, of either sign)
    and float32 sums of up to 4200 terms (2^-24 sqrt(4200) = 4e-6) by less than the bounds.  (The normalised dq is a difference of nearly equal
    sums, which bfloat16's rounding has no such bound for.)"""
    print(f"case long scans {shape} {dtype} {p}", flush=True)
    q, k, v, gate, do, done, S0, z0, dS, dz, _ = _inputs(shape, dtype, p, True, 9)
    for normalise in (False, True) if dtype == "f32" else (False,):
        leaves = [t.detach().requires_grad_() for t in ((q, k, v, S0, z0) if normalise else (q, k, v, gate, S0))]
        cotangents = (do, dS, dz) if normalise else (do, dS)
        if normalise:
            yard = _exact_with_gradients((q, k, v, None, S0, z0), done, "elu1", True, cotangents)
            out = Fn.normalised_linear_attention(*leaves[:3], done, *leaves[3:], "elu1")[:3]
        else:
            yard = _exact_with_gradients((q, k, v, gate, S0, None), done, "elu1", False, cotangents)
            out = Fn.gated_linear_attention(*leaves[:4], done, leaves[4], "elu1")
        for x, y in zip((*out, *torch.autograd.grad(out, leaves, cotangents)), sum(yard, [])):
            assert _distance(x, y) <= (1e-2 if dtype == "bf16" else 1e-5), (normalise, tuple(x.shape), _distance(x, y))


@pytest.mark.parametrize("form", ["gated", "normalised"])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_what_lies_before_a_reset_reaches_nothing_after_it(form, dtype):
    q, k, v, gate, do, done, S0, z0, dS, dz, _ = _inputs((2, 1, 64, 64, 9.3), dtype, 0.0, True, 7)
    at = q.shape[1] // 2 + 5
    done[:, at] = True
    with torch.no_grad():
        for t in (q, k, v, gate):
            t[:, at - 20:at - 10] = float("nan")
    leaves = [t.requires_grad_() for t in (q, k, v)]
    if form == "gated":
        o, S = Fn.gated_linear_attention(q, k, v, gate, done, S0, "elu1")
        grads = torch.autograd.grad((o, S), leaves, (do, dS))
    else:
        o, S, z = Fn.normalised_linear_attention(q, k, v, done, S0, z0, "elu1")[:3]
        grads = torch.autograd.grad((o, S, z), leaves, (do, dS, dz))
    for t in (o, *grads):
        assert torch.isfinite(t[:, at:]).all()
    assert torch.isfinite(S).all()
