"""Columns of a panel at scales whose products leave the range of a double, where no
column's own sum of squares tells it: the last column of a square panel, and the
columns that the DM truncation rejects.  Each column to its own scale."""
import numpy as np
import pytest

from test_gpu_regpanel import gpu, lapack, qrf  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 64, 128, 200])
@pytest.mark.parametrize("first,last", [(1e-130, 1e-200), (1e-139, 1e-185), (1e130, 1e200)])
def test_last_column_of_a_square(gpu, n, first, last):  # noqa: F811
    print("panel scales", n, first, last, flush=True)
    a = np.random.default_rng(n).standard_normal((n, n)) * first
    a[:, -1] *= last / first
    (g, _), (b, _) = qrf(gpu, a), lapack(a)
    for c, s in ((slice(0, n - 1), first), (slice(n - 1, n), last)):
        d = np.triu(g)[:, c] / s - np.triu(b)[:, c] / s
        assert np.linalg.norm(d) <= 1e-12 * np.linalg.norm(a[:, c] / s), s


@pytest.mark.parametrize("m", [100, 400])
def test_rejected_columns(gpu, oracle, m):  # noqa: F811
    import qrdm_amd
    n = 12
    a = np.random.default_rng(m).standard_normal((m, n)) * 1e-200
    a[:, -1] *= 1e70  # the walk puts the last column first
    print("panel scales, rejected", m, flush=True)
    ref = oracle.dgeqrdm(a, tau=0.0)
    d = gpu.from_numpy(np.ascontiguousarray(a.T)).cuda()
    tau = gpu.zeros(n, dtype=gpu.float64, device="cuda")
    jp, nc = np.zeros(n, np.int32), np.zeros(n, np.int32)
    info, _ = qrdm_amd.dgeqrdm_dev(d, m, tau, jp, nc, np.array([0.9, 0.0, 0.0]))
    assert info == 0 and jp[0] == n and ref["jpvt"][0] == n
    # the first row: one reflection, columns in any order after it
    r = np.zeros(n)
    r[jp - 1] = d.cpu().numpy()[:, 0]
    rr = np.zeros(n)
    rr[ref["jpvt"] - 1] = ref["a"][0]
    assert np.abs(r - rr)[:-1].max() <= 1e-12 * 1e-200 * np.sqrt(m)
