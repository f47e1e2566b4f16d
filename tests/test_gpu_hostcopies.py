"""Host-pointer entry points: packed and strided blocks give the same factors,
and what lies between the columns of a strided block is left alone."""
import ctypes

import numpy as np
import pytest

import qrdm_amd

pytestmark = pytest.mark.gpu


def strided(x, ld):
    buf = np.full((x.shape[1], ld), 7.25)
    buf[:, : x.shape[0]] = x.T
    return buf


def ptr(x, t=ctypes.c_double):
    return x.ctypes.data_as(ctypes.POINTER(t))


# one row, one column, odd sizes, and blocks of more than one staged chunk
# (8 MB: 2100 x 501 doubles are 8.4 MB, three columns of 400001 are 9.6 MB)
@pytest.mark.parametrize("m,n", [(1, 5), (7, 1), (37, 53), (130, 61), (2100, 501), (400001, 3)])
def test_strided_equals_packed(m, n):
    assert pytest.importorskip("torch").cuda.is_available(), "-m gpu run without a GPU"
    lib = qrdm_amd.lib()
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n))
    c = rng.standard_normal((m, 3))
    k = min(m, n)
    out = []
    for ld in (m, m + 5):
        buf, jp, tau = strided(a, ld), np.zeros(n, np.int32), np.zeros(k)
        ncols, thres = np.zeros(n + 1, np.int32), np.array([0.9, 0.15, 0.0])
        info = lib.dgeqrdm(102, m, n, ptr(buf), ld, ptr(jp, ctypes.c_int), ptr(tau),
                           ptr(ncols, ctypes.c_int), ptr(thres), 32)
        qr, qtau, cb = strided(a, ld), np.zeros(k), strided(c, ld)
        info2 = lib.qrdm_dgeqrf(m, n, ptr(qr), ld, ptr(qtau))
        info3 = lib.qrdm_dormqr(1, m, 3, k, ptr(qr), ld, ptr(qtau), ptr(cb), ld)
        assert (info, info2, info3) == (0, 0, 0)
        for x in (buf, qr, cb):
            assert (x[:, m:] == 7.25).all()
        out.append((buf[:, :m], jp, tau, ncols, qr[:, :m], qtau, cb[:, :m]))
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
