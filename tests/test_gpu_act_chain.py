"""Stacks that act in one native call (stack_act: act_chain.hip between the state updates) against the same blocks one by one, and the kernels at the
edges of their tiles: 16 rows, 16 columns of a wave, 128 bytes of a weight row, workgroups of 64 and 256 columns, rows up to and past those that are chained."""
import ctypes

import pytest
import torch

from gpu_util import relerr

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def _np(t):
    return t.detach().float().cpu().numpy()


def _model(kinds, F, H, d, norm, dtype=BF):
    from memorax_amd import sequence_models as sm
    torch.manual_seed(F + H + d)
    make = {"delta": lambda: sm.Memoroid(sm.DeltaNetCell(F, d, H, dtype=dtype)), "linear": lambda: sm.Memoroid(sm.LinearAttentionCell(F, d, H)),
            "gated": lambda: sm.GatedLinearRecurrence(F), "wide": lambda: sm.GatedLinearRecurrence(F, hidden=F + 24),
            "lru": lambda: sm.Memoroid(sm.LRUCell(F, 32))}
    with torch.device("cuda"):
        m = sm.Stack([sm.Residual(sm.PreNorm(make[k](), F, norm=norm)) for k in kinds]).cuda()
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 1:
                p.add_(torch.randn_like(p) * 0.3)
    return m


def _leaves(t):
    return [t] if torch.is_tensor(t) else [x for v in t for x in _leaves(v)]


@pytest.mark.parametrize("kinds", [("delta", "gated", "delta", "gated"), ("linear", "linear", "wide"), ("gated", "lru", "delta"), ("wide", "gated")])
@pytest.mark.parametrize("B,F,H,d", [(1, 8, 1, 8), (17, 64, 2, 16), (33, 72, 2, 24), (130, 136, 3, 40), (1024, 256, 4, 64), (1030, 256, 8, 64), (16, 264, 2, 32),
                                     (4096, 64, 2, 16), (4097, 64, 2, 16)])   # a workgroup for each compute unit, and one more
@pytest.mark.parametrize("rms,autocast", [(True, True), (False, True), (True, False)])
def test_stack_acts_as_its_blocks(kinds, B, F, H, d, rms, autocast):
    from memorax_amd import sequence_models as sm
    from memorax_amd.functional import step_in_place
    if B > 1000 and kinds[0] != "delta":
        pytest.skip("the largest rows once")
    m = _model(kinds, F, H, d, sm.RMSNorm if rms else sm.LayerNorm, BF if d % 8 == 0 else F32)
    g = torch.Generator(device="cuda").manual_seed(B)
    carry, want_carry = m.initialize_carry(None, (B, F)), None
    want_carry = carry
    tol = 2e-2 if autocast or "delta" in kinds else 1e-4   # bfloat16 of a sum the other way, through up to four blocks; float32 sums in another order
    print(f"case stack {kinds} {B} {F} {H} {d} {rms} {autocast}", flush=True)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=autocast):
        for t in range(3):
            x = torch.randn(B, 1, F, device="cuda", generator=g)
            done = torch.rand(B, 1, device="cuda", generator=g) < 0.2
            kept = [c.clone() for c in _leaves(carry)]
            held = carry
            carry, y = m(x, done, carry)
            assert all(torch.equal(a, b) for a, b in zip(kept, _leaves(held)))   # not in place
            want, nexts = x, []
            for block, c in zip(m.blocks, want_carry):
                c, want = block(want, done=done, initial_carry=c)
                nexts.append(c)
            want_carry = tuple(nexts)
            assert relerr(y, _np(want)) <= tol
            for a, b in zip(_leaves(carry), _leaves(want_carry)):
                assert a.shape == b.shape and a.dtype == b.dtype
                if not a.is_complex():
                    assert relerr(a.exp() if a.dim() == 3 else a, _np(b.exp() if a.dim() == 3 else b)) <= 2 * tol
        with step_in_place():
            mine = [c.clone() for c in _leaves(carry)]
            again, y2 = m(x, done, carry)
            apart, _ = m(x, done, _tree(carry, iter(mine)))
        if "lru" not in kinds:
            assert all(a.data_ptr() == b.data_ptr() for a, b in zip(_leaves(again), _leaves(carry)))
            assert all(torch.equal(a, b) for a, b in zip(_leaves(again), _leaves(apart)))


def _tree(like, it):
    return next(it) if torch.is_tensor(like) else tuple(_tree(v, it) for v in like)


def test_a_stack_of_other_blocks_asks_nothing_of_its_own(monkeypatch):
    from memorax_amd import sequence_models as sm
    m = _model(("lru", "lru"), 64, 2, 16, sm.RMSNorm, F32)
    asked, of = [], sm._acting_rows
    monkeypatch.setattr(sm, "_acting_rows", lambda x: asked.append(1) or of(x))
    monkeypatch.setattr(sm, "_run_of_blocks", None)
    with torch.no_grad():
        m(torch.randn(4, 1, 64, device="cuda"), torch.zeros(4, 1, dtype=torch.bool, device="cuda"), m.initialize_carry(None, (4, 64)))
    assert len(asked) == 2   # each block for itself


def test_hook_in_a_block_is_run():
    from memorax_amd import sequence_models as sm
    m, seen = _model(("delta", "gated", "delta"), 64, 2, 16, sm.RMSNorm), []
    x, done = torch.randn(4, 1, 64, device="cuda"), torch.zeros(4, 1, dtype=torch.bool, device="cuda")
    m.blocks[1].module.module.out.register_forward_hook(lambda *a: seen.append(1))
    with torch.no_grad():
        carry, _ = m(x, done)
    assert seen == [1] and len(carry) == 3


class _Closing(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("rows", "scale", "weight", "bias", "residual", "out")] + [("K", ctypes.c_int64)] + \
               [(n, ctypes.c_int) for n in ("norm", "round_norm", "row_dtype", "bias_dtype")] + [("eps", ctypes.c_float)]


@pytest.mark.parametrize("rows,K,F,ns", [(1, 8, 8, (8,)), (15, 24, 56, (16, 17, 3)), (16, 512, 64, (64, 64, 64, 2)), (17, 72, 128, (256, 4)), (33, 264, 136, (300, 5, 40)),
                                         (49, 256, 256, (256, 256, 256, 4)), (16, 256, 248, (1024, 8))])
@pytest.mark.parametrize("wd,product,xd", [(F32, F32, F32), (F32, BF, BF), (BF, BF, BF), (BF, BF, F32)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_closed_row_dense(rows, K, F, ns, wd, product, xd, norm):
    from memorax_amd import _lib
    lib, n = _lib.load(), _lib.native()
    g = torch.Generator(device="cuda").manual_seed(rows + K + F)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    code = lambda dt: 0 if dt == F32 else 1  # noqa: E731
    h, res = rand(rows, 1, K).to(xd), rand(rows, 1, F)
    cs, cw, cb = rand(K), (rand(F, K) * K ** -0.5).to(wd), rand(F).to(BF if norm == 1 else F32)
    scale, nbias = rand(F) if norm else None, rand(F) if norm == 2 else None
    ws = [(rand(o, F) * F ** -0.5).to(wd) for o in ns]
    bs = [rand(o) if i % 2 == 0 else None for i, o in enumerate(ns)]
    want_x = n.row_dense(h, norm % 2, cs if norm % 2 else None, None, 1e-6, xd == BF, [cw], [cb], product, F32, res)[0]
    want = n.row_dense(want_x, norm, scale, nbias, 1e-5, False, ws, bs, product, xd, None)
    out = torch.full_like(want_x, float("nan"))
    ys = [torch.full_like(t, float("nan")) for t in want]
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    c = _Closing(p(h), p(cs) if norm % 2 else None, p(cw), p(cb), p(res), p(out), K, norm % 2, xd == BF, code(xd), code(cb.dtype), 1e-6)
    arr = lambda v: (ctypes.c_void_p * len(v))(*v)  # noqa: E731
    print(f"case closed {rows} {K} {F} {ns} {wd} {product} {xd} {norm}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    rc = lib.mrx_closed_row_dense(stream, ctypes.byref(c), p(scale), p(nbias), norm, arr([p(w) for w in ws]), arr([p(b) for b in bs]), arr([p(y) for y in ys]),
                                  (ctypes.c_int64 * len(ns))(*ns), len(ns), rows, F, code(wd), 0, code(xd), code(product), 1e-5)
    torch.cuda.synchronize()
    assert rc == 0
    # float32 sums of up to 512 products in another order; with bfloat16 roundings behind them a result may round the other way
    tol = 1e-5 if product == F32 and xd == F32 else 1e-2
    assert relerr(out, _np(want_x)) <= tol
    for y, w in zip(ys, want):
        assert relerr(y, _np(w)) <= tol


@pytest.mark.parametrize("rows,K,F,N", [(1, 8, 8, 8), (15, 24, 56, 60), (16, 512, 64, 64), (17, 72, 128, 200), (33, 264, 136, 68), (49, 256, 256, 256), (16, 512, 256, 512),
                                        (1040, 128, 128, 256)])   # the last: two workgroups on a compute unit
@pytest.mark.parametrize("wd,product", [(F32, F32), (F32, BF), (BF, BF)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_closed_gated_recurrence(rows, K, F, N, wd, product, norm):
    """The closing layer and the gated step in one launch against the row kernel and then the gated step alone."""
    from memorax_amd import _lib
    lib, n = _lib.load(), _lib.native()
    g = torch.Generator(device="cuda").manual_seed(rows + K + F + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    code = lambda dt: 0 if dt == F32 else 1  # noqa: E731
    h, res = rand(rows, 1, K).to(product), rand(rows, 1, F)
    cs, cw, cb = rand(K), (rand(F, K) * K ** -0.5).to(wd), rand(F)
    scale, nbias = rand(F) if norm else None, rand(F) if norm == 2 else None
    ws = [(rand(N, F) * F ** -0.5).to(wd) for _ in range(3)]
    done = torch.rand(rows, 1, device="cuda", generator=g) < 0.3
    ls, ld = rand(rows, 1, N), -torch.rand(rows, 1, N, device="cuda", generator=g)
    ls[0] = -float("inf")   # a carry of zero
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    st = torch.cuda.current_stream().cuda_stream
    fresh = lambda: [torch.full((rows, 1, N), float("nan"), device="cuda", dtype=dt) for dt in (product, product, F32, F32)]  # noqa: E731
    print(f"case closed gated {rows} {K} {F} {N} {wd} {product} {norm}", flush=True)
    want_x = n.row_dense(h, norm % 2, cs if norm % 2 else None, None, 1e-6, product == BF, [cw], [cb], product, F32, res)[0]
    want, got, out = fresh(), fresh(), torch.full_like(want_x, float("nan"))
    tail = lambda o: (*(p(w) for w in ws), p(done), p(ls), p(ld), *(p(t) for t in o), rows, F, N, code(wd), code(product), 0, 1e-5)  # noqa: E731
    assert lib.mrx_gated_recurrence_act(st, p(want_x), p(scale), p(nbias), norm, *tail(want)) == 0
    c = _Closing(p(h), p(cs) if norm % 2 else None, p(cw), p(cb), p(res), p(out), K, norm % 2, product == BF, code(product), 0, 1e-6)
    assert lib.mrx_closed_gated_recurrence_act(st, ctypes.byref(c), None, p(scale), p(nbias), norm, *tail(got)) == 0
    torch.cuda.synchronize()
    # each on its own scale: x' as above; z, the gated state and the state's exponential behind one more product of up to 256 terms and its roundings
    tol = 1e-5 if product == F32 else 1e-2
    assert relerr(out, _np(want_x)) <= tol
    for a, b in ((got[0], want[0]), (got[1], want[1]), (got[2].exp(), want[2].exp()), (got[3], want[3])):
        assert relerr(a, _np(b)) <= 2 * tol
