"""The row slabs of a merged trailing pass, chosen on the host and, with the same
function, in two kernels that have to agree: the least whole-number cost, the
fewest slabs among equals."""
import ctypes

import pytest

import qrdm_amd


def expected(m, n, ncol):
    nchunk, groups = -(-m // 32), -(-ncol // 64)
    best = None
    for ns in range(1, 65):
        per = -(-ns * groups // 8)
        if ns > 1 and (per > 64 or ns > nchunk or ns * ncol > 16 * n):
            continue
        cost = (34 if per > 32 else 20) * (-(-nchunk // ns) + 2) + ns
        if best is None or cost < best[0]:
            best = (cost, ns)
    return best[1]


@pytest.mark.parametrize("m,n,c0", [
    (72608, 1792, 1344), (72640, 1792, 1344),  # 36 and 64 slabs cost the same
    (1, 2, 1), (33, 100, 1), (8192, 8192, 64), (16384, 1024, 64), (3001, 1777, 500), (64, 40000, 1)])
def test_slabs(m, n, c0):
    f = ctypes.CDLL(qrdm_amd.LIB_PATH)._ZN4qrdm11fused_slabsEiiii
    assert f(0, m, c0, n) == expected(m, n, n - c0)
