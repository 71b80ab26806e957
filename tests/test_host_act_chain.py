"""What the acting chain's entry points refuse, without a GPU: nothing is launched, the addresses are never read."""
import pytest

INVALID, UNSUPPORTED = -1, -2
AT = [(i + 1) << 24 for i in range(32)]   # addresses of arrays, sixteen megabytes apart


@pytest.mark.parametrize("K,N,status", [(12, 64, INVALID), (508, 64, INVALID), (0, 64, INVALID), (516, 64, UNSUPPORTED), (520, 64, UNSUPPORTED), (64, 6, UNSUPPORTED)])
def test_gated_step_tells_what_is_wrong_from_what_is_not_covered(K, N, status):
    """Features that are no multiple of eight are invalid, as for the row kernels; more than a workgroup holds is not covered."""
    from memorax_amd import _lib
    p = AT
    assert _lib.load().mrx_gated_recurrence_act(None, p[0], p[1], None, 1, p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11], 16, K, N, 0, 1, 0, 1e-6) == status
