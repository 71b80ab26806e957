"""The diagonal scans where the plan changes: rows that are no whole number of vectors (also narrower than one), super-steps of
16 steps per wave and their remainders, streaming kernels on ragged rows, time in segments; every kind of array, forward and backward, against a
sequential reference in double precision."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [
    (2, 257, 1), (3, 130, 3), (2, 256, 5),        # rows narrower than a vector, sixteen waves and a remainder
    (3, 40, 131), (2, 128, 129), (70, 66, 191),   # a last tile of one or a few lanes
    (2, 513, 65), (5, 272, 130),
    (300, 520, 70),                               # eight waves of 16 steps
    (1101, 33, 131), (601, 65, 257),              # streaming on ragged rows
    (135, 515, 200), (300, 70, 256),              # bfloat16: more workgroups than one or two per compute unit
    (1, 385, 2), (1, 513, 65), (12, 450, 130), (1, 1200, 512),   # time in segments, the last one partly filled
    (1, 4096, 70),                                # as many segments as there can be
]


def _reference(kind, a, b, done, h0, g, gl):
    """h, h_last and the gradients of sum(g h) + sum(gl h_last) in double precision on the device."""
    wide = torch.complex128 if a.is_complex() else torch.float64
    a, b, h0 = (x.detach().to(wide).requires_grad_() for x in (a, b, h0))
    if kind == "mingru":
        keep, inp = torch.sigmoid(-a), torch.sigmoid(a) * torch.where(b >= 0, b + 0.5, torch.sigmoid(b))
    else:
        keep, inp = a, b
    h, out = h0, []
    for t in range(b.shape[1]):
        k = keep if a.ndim == 1 else keep[:, t]
        h = torch.where(done[:, t, None], 0.0, k * h) + inp[:, t]
        out.append(h)
    hs = torch.stack(out, 1)
    grads = torch.autograd.grad([hs, h], [a, b, h0], [g.to(wide), gl.to(wide)])
    return [x.detach() for x in (hs, h, *grads)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["f32", "bf16", "c64", "c64 broadcast", "mingru", "mingru bf16"])
def test_scan_plans(kind, shape):
    from memorax_amd import kernels as K
    B, T, D = shape
    gen = torch.Generator(device="cuda").manual_seed(B + 3 * T + 7 * D)
    half = "bf16" in kind
    E = torch.complex64 if "c64" in kind else torch.float32
    S = torch.bfloat16 if half else E
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=E)
    a_shape = (D,) if "broadcast" in kind else shape
    a = rnd(*a_shape)
    if "mingru" not in kind:
        a = 0.95 * a / a.abs() if E.is_complex else torch.rand(a_shape, generator=gen, device="cuda") * 0.2 + 0.8
    a, b, g, h0, gl = a.to(S), rnd(*shape).to(S), rnd(*shape).to(S), rnd(B, D), rnd(B, D)
    done = torch.rand(B, T, generator=gen, device="cuda") < 0.02
    print(f"case scan plans {kind} {shape}", flush=True)
    mingru = "mingru" in kind
    h, hl, _ = (K.mingru_scan_fwd if mingru else K.linear_scan_fwd)(a, b, done, h0)
    if mingru:
        da, db, dh0 = K.mingru_scan_bwd(a, b, h, done, h0, g, gl)
    else:
        da, db, dh0 = K.linear_scan_bwd(a, h, done, h0, g, gl, sum_da="broadcast" in kind)
        da = da.sum(0) if "broadcast" in kind else da
    ref = _reference("mingru" if mingru else "linear", a, b, done, h0, g, gl)
    for name, x, r, tol in zip(("h", "h_last", "da", "db", "dh0"), (h, hl, da, db, dh0), ref,
                               (2e-2, 1e-4, 2e-2, 2e-2, 2e-2) if half else (1e-4,) * 5):
        err = float((x.to(r.dtype) - r).abs().max() / r.abs().max().clamp_min(1e-30))
        assert err <= tol, (name, err)


WIDE = [
    (405, 66, 176), (403, 67, 200), (410, 65, 201),      # four waves on wide vectors: whole and ragged rows, spans partly filled
    (1100, 64, 256), (1101, 70, 257),                    # whole rows streaming on wide vectors (MinGRU, bfloat16)
    (520, 70, 100), (520, 72, 256), (260, 80, 128),      # two elements and single ones per lane, four waves
    (405, 97, 67), (134, 101, 515),                      # a lane of the last tile
    (1025, 513, 256), (130, 1009, 1024), (260, 520, 1000),   # large float32 calls (2^27 elements and more)
]


@pytest.mark.parametrize("shape", WIDE)
@pytest.mark.parametrize("kind", ["f32", "f32 broadcast", "bf16", "bf16 broadcast", "c64", "c64 broadcast", "mingru", "mingru bf16"])
def test_wide_splits(kind, shape):
    if shape[0] * shape[1] * shape[2] >= 1 << 27 and kind not in ("f32", "mingru"):
        pytest.skip("float32 storage with coefficients of every step only")
    test_scan_plans(kind, shape)
