"""Dense layers on few rows with the norm before and the residual behind (mrx_row_dense), the MinGRU and DeltaNet acting steps,
and the pre-norm residual blocks that act through them, against array operations."""
import pytest
import torch
import torch.nn.functional as F

from gpu_util import relerr

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def _np(t):
    return t.detach().float().cpu().numpy()


@pytest.mark.parametrize("rows,K,ns", [
    (1, 8, [1]), (15, 24, [3, 64]), (16, 256, [64, 63, 4]), (33, 264, [65]), (100, 520, [200, 5, 17, 128]), (513, 256, [256, 256, 256, 4]),
    (2050, 512, [100]), (7, 1032, [40]), (4, 2048, [12])])
@pytest.mark.parametrize("xd,wd,product,out", [(F32, F32, F32, F32), (F32, F32, BF, BF), (BF, BF, BF, BF), (F32, BF, BF, F32), (BF, F32, F32, BF)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_row_dense_against_array_operations(rows, K, ns, xd, wd, product, out, norm):
    from memorax_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows + K)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x = rand(rows, 1, K).to(xd)
    scale, nbias = rand(K), rand(K)
    ws = [(rand(n, K) / K ** 0.5).to(wd) for n in ns]
    bs = [rand(n) if i % 2 == 0 else None for i, n in enumerate(ns)]
    residual = rand(rows, 1, ns[0]) if len(ns) == 1 else None
    od = F32 if residual is not None else out
    print(f"case rows {rows} {K} {ns} {xd} {wd} {product} {norm}", flush=True)
    got = _lib.native().row_dense(x, norm, scale if norm else None, nbias if norm == 2 else None, 1e-6, xd == BF, ws, bs, product, od,
                                  residual)
    h = x.double()
    if norm == 1:
        h = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6) * scale.double()
    elif norm == 2:
        h = F.layer_norm(h, (K,), scale.double(), nbias.double(), 1e-6)
    if product == BF or (norm and xd == BF):
        h = h.float().to(BF)
    for y, w, b in zip(got, ws, bs):
        w, b = (w.to(BF), None if b is None else b.to(BF)) if product == BF else (w, b)
        ref = F.linear(h.double(), w.double(), None if b is None else b.double())
        if residual is not None:
            ref = ref + residual.double()
        assert y.dtype == od and y.shape == ref.shape
        tol = 1e-5 if product == F32 and od == F32 and not (norm and xd == BF) else 2e-2
        assert relerr(y, _np(ref)) <= tol, relerr(y, _np(ref))


@pytest.mark.parametrize("B,D,dtype", [(1, 1, F32), (3, 5, F32), (70, 256, BF), (33, 12, F32), (5, 7, BF)])
def test_mingru_step_against_the_scan(B, D, dtype):
    from memorax_amd import _lib
    from memorax_amd import functional as Fn
    g = torch.Generator(device="cuda").manual_seed(B * D)
    z, x, gate = (torch.randn(B, 1, D, device="cuda", generator=g).to(dtype) for _ in range(3))
    done = torch.rand(B, 1, device="cuda", generator=g) < 0.3
    ls, ld = torch.randn(B, 1, D, device="cuda", generator=g), -torch.rand(B, 1, D, device="cuda", generator=g)
    if B > 1:
        ls[1] = -float("inf")
    h, h_last, P_last = Fn.mingru_scan(z, x, done, ls[:, 0].exp(), ld[:, 0].exp())
    want = (h.float() * F.silu(gate.float())).to(dtype)
    tol = 1e-5 if dtype == F32 else 1e-2
    for in_place in (False, True):
        a, b = ls.clone(), ld.clone()
        y, s, d = _lib.native().mingru_step(z, x, gate, done, a, b, in_place)
        assert (s.data_ptr() == a.data_ptr()) == in_place
        assert relerr(y, _np(want)) <= tol
        assert relerr(s[:, 0].exp(), _np(h_last)) <= 1e-5 and relerr(d[:, 0].exp(), _np(P_last)) <= 1e-5
    y, _, _ = _lib.native().mingru_step(z, x, None, done, ls, ld, False)
    assert relerr(y, _np(h)) <= tol


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("autocast", [False, True])
def test_acting_blocks_equal_their_composition(d, autocast):
    """With gradients enabled a block runs its composition; without, at T = 1, the fused acting step."""
    from memorax_amd import sequence_models as sm
    torch.manual_seed(d)
    B, Fe, H = 37, 64, 2
    cells = [sm.Memoroid(sm.DeltaNetCell(Fe, d, H)), sm.Memoroid(sm.DeltaNetCell(Fe, d, H, dtype=F32)), sm.GatedLinearRecurrence(Fe, 40),
             sm.Memoroid(sm.LinearAttentionCell(Fe, d, H)), sm.Memoroid(sm.MambaCell(Fe, H, d, d))]
    for cell in cells[:4] if autocast else cells:
        for norm in (sm.RMSNorm, sm.LayerNorm):
            block = sm.Residual(sm.PreNorm(cell, Fe, norm=norm)).cuda()
            carry = ref = block.initialize_carry(None, (B, Fe))
            for t in range(3):
                x, done = torch.randn(B, 1, Fe, device="cuda"), torch.rand(B, 1, device="cuda") < 0.3
                with torch.autocast("cuda", dtype=BF, enabled=autocast):
                    ref, want = block(x, done, ref)
                    with torch.no_grad():
                        carry, y = block(x, done, carry)
                tol = 2e-2 if autocast or isinstance(getattr(cell, "cell", None), sm.DeltaNetCell) else 1e-4
                name = f"{type(cell).__name__} {type(getattr(cell, 'cell', cell)).__name__} {norm} {t}"
                assert y.dtype == want.dtype and relerr(y, _np(want)) <= tol, (name, relerr(y, _np(want)))
                for a, b in zip(carry, ref):
                    assert a.shape == b.shape and a.dtype == b.dtype and relerr(a, _np(b)) <= tol, (name, relerr(a, _np(b)))
                ref = tuple(c.detach() for c in ref)


@pytest.mark.parametrize("cell", ["lru 8", "lru 136", "mlstm 1 16", "mlstm 3 16", "mlstm 8 32", "mlstm 2 64", "mlstm 4 64"])
@pytest.mark.parametrize("B", [1, 45])
def test_acting_lru_and_mlstm_blocks_equal_their_composition(cell, B):
    from memorax_amd import sequence_models as sm
    torch.manual_seed(B)
    Fe = 72
    kind, *sizes = cell.split()
    sizes = [int(s) for s in sizes]
    make = (lambda: sm.LRUCell(Fe, *sizes)) if kind == "lru" else (lambda: sm.mLSTMCell(Fe, hidden_dim=sizes[0] * sizes[1], num_heads=sizes[0]))
    for norm in (sm.RMSNorm, sm.LayerNorm):
        block = sm.Residual(sm.PreNorm(sm.Memoroid(make()), Fe, norm=norm)).cuda()
        with torch.no_grad():   # initial zeros would hide a wrong index
            for p in block.parameters():
                p.add_(0.1 * torch.randn_like(p))
        if kind == "lru":
            block.module.module.cell.gamma_log.data.clamp_(max=0.3)
        carry = ref = block.initialize_carry(None, (B, Fe))
        for t in range(4):
            x, done = torch.randn(B, 1, Fe, device="cuda"), torch.rand(B, 1, device="cuda") < 0.3
            ref, want = block(x, done, ref)
            with torch.no_grad():
                carry, y = block(x, done, carry)
            assert y.dtype == want.dtype and relerr(y, _np(want)) <= 1e-4, (t, relerr(y, _np(want)))
            for a, b in zip(carry, ref):
                assert a.shape == b.shape and a.dtype == b.dtype
                a, b = (torch.view_as_real(v.detach().contiguous()) if v.is_complex() else v.detach() for v in (a, b))
                assert relerr(a, _np(b)) <= 1e-4, (t, relerr(a, _np(b)))
            ref = tuple(c.detach() for c in ref)


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("rows,K,n,own", [(1024, 512, 512, True), (1025, 512, 512, False), (4096, 256, 256, True), (4097, 256, 256, False),
                                          (16384, 64, 256, True), (16385, 64, 64, False), (9, 520, 16, False), (16384, 1024, 512, False),
                                          (256, 2048, 64, False)])
def test_dense_layers_take_the_row_kernel_up_to_its_line(rows, K, n, own, autocast):
    """Beyond the line the array library's products, bit for bit; up to it one launch, whose sums run in another order."""
    from memorax_amd.dense import Weights, dense_group
    from memorax_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, K, device="cuda", generator=g)
    layers = [Weights(torch.randn(n, K, device="cuda", generator=g) / K ** 0.5, torch.randn(n, device="cuda", generator=g) if i else None)
              for i in range(2)]
    assert _lib.native().rows_pay(rows, K, 2 * n * K, 2, False, autocast) == own
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=autocast):
        got = dense_group(x, layers)
        want = [F.linear(x, w, b) for w, b in layers]
    for y, w, (weight, bias) in zip(got, want, layers):
        assert y.dtype == w.dtype
        if not own:
            assert torch.equal(y, w)
        else:
            ops = [t.to(BF).double() if autocast else t.double() for t in (x, weight)]
            ref = F.linear(*ops, None if bias is None else bias.to(BF).double() if autocast else bias.double())
            assert relerr(y, _np(ref)) <= (2e-2 if autocast else 1e-5)


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("rows,Fe,own", [(1024, 512, True), (1025, 512, False), (128, 1024, True), (129, 1024, False), (32, 2048, None), (33, 2048, False)])
def test_acting_blocks_around_their_line(rows, Fe, own, autocast):
    from memorax_amd import sequence_models as sm
    torch.manual_seed(rows)
    own = autocast if own is None else own   # rows of 2048 features: bfloat16 products only
    block = sm.Residual(sm.PreNorm(sm.GatedLinearRecurrence(Fe), Fe)).cuda()
    x, done = torch.randn(rows, 1, Fe, device="cuda"), torch.rand(rows, 1, device="cuda") < 0.3
    with torch.autocast("cuda", dtype=BF, enabled=autocast):
        with torch.no_grad():
            assert (block.module.module.acting(x, block.module.norm, done, None) is not None) == own
            carry, y = block(x, done)
        ref, want = block(x, done)
    assert y.dtype == want.dtype
    for a, b in zip([y, *carry], [want, *ref]):
        assert relerr(a, _np(b)) <= (2e-2 if autocast else 1e-4)
