"""What the acting chain's entry points refuse, without a GPU: nothing is launched, the addresses are never read."""
import ctypes

import pytest

INVALID, UNSUPPORTED = -1, -2
AT = [(i + 1) << 24 for i in range(32)]   # addresses of arrays, sixteen megabytes apart


@pytest.mark.parametrize("K,N,status", [(12, 64, INVALID), (508, 64, INVALID), (0, 64, INVALID), (516, 64, UNSUPPORTED), (520, 64, UNSUPPORTED), (64, 6, UNSUPPORTED)])
def test_gated_step_tells_what_is_wrong_from_what_is_not_covered(K, N, status):
    """Features that are no multiple of eight are invalid, as for the row kernels; more than a workgroup holds is not covered."""
    from memorax_amd import _lib
    p = AT
    assert _lib.load().mrx_gated_recurrence_act(None, p[0], p[1], None, 1, p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11], 16, K, N, 0, 1, 0, 1e-6) == status


class _Closing(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("rows", "scale", "weight", "bias", "residual", "out")] + [("K", ctypes.c_int64)] + \
               [(n, ctypes.c_int) for n in ("norm", "round_norm", "row_dtype", "bias_dtype")] + [("eps", ctypes.c_float)]


@pytest.mark.parametrize("out,status", [("residual", INVALID), ("residual's last row", INVALID), ("before residual, one row over", INVALID), ("rows", INVALID),
                                        ("rows' last", INVALID), ("behind residual", UNSUPPORTED), ("behind rows", UNSUPPORTED)])
@pytest.mark.parametrize("gated", [False, True])
def test_a_closing_layer_may_not_write_what_it_reads(out, status, gated):
    """Other workgroups of a row tile still read the residual and the rows when the first writes the result.  (What passes is told by the answer to the next check:
    openings wider than 2^24 columns are not covered.)"""
    from memorax_amd import _lib
    R, F, K, p = 48, 64, 128, AT
    at = {"residual": p[4], "residual's last row": p[4] + (R - 1) * F * 4, "before residual, one row over": p[4] - (R - 1) * F * 4, "rows": p[0], "rows' last": p[0] + (R - 1) * K * 2,
          "behind residual": p[4] + R * F * 4, "behind rows": p[0] + R * K * 2}[out]
    c, wide = _Closing(p[0], p[1], p[2], p[3], p[4], at, K, 1, 0, 1, 0, 1e-6), (1 << 24) + 4
    arr = lambda *v: (ctypes.c_void_p * len(v))(*v)  # noqa: E731
    if gated:
        rc = _lib.load().mrx_closed_gated_recurrence_act(None, ctypes.byref(c), None, p[6], None, 1, p[7], p[8], p[9], p[10], p[11], p[12], p[13], p[14], p[15], p[16], R, F, wide,
                                                         0, 1, 0, 1e-6)
    else:
        rc = _lib.load().mrx_closed_row_dense(None, ctypes.byref(c), p[6], None, 1, arr(p[7]), arr(None), arr(p[8]), (ctypes.c_int64 * 1)(wide), 1, R, F, 0, 0, 0, 1, 1e-6)
    assert rc == status
