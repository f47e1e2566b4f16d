"""Q applied from given reflectors (ormqr): block and tile edges, both
directions, any leading dimension, zero tau, against the reflectors applied one
by one in extended precision."""
import numpy as np
import pytest

import qrdm_amd

pytestmark = pytest.mark.gpu


def apply_reflectors(a, tau, c, trans):
    c = c.astype(np.longdouble)
    m, k = a.shape[0], len(tau)
    for i in range(k) if trans else reversed(range(k)):
        v = np.zeros(m, np.longdouble)
        v[i], v[i + 1:] = 1, a[i + 1:, i]
        c -= np.longdouble(tau[i]) * np.outer(v, v @ c)
    return c


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("m,n,k,pad", [
    (1, 1, 1, 0), (40, 3, 1, 1), (64, 16, 64, 0), (65, 17, 65, 3), (127, 64, 63, 0),
    (200, 65, 128, 1), (333, 130, 191, 2), (700, 31, 449, 0), (2500, 70, 70, 5), (2100, 1500, 129, 0)])
def test_ormqr_edges(m, n, k, pad, trans):
    torch = pytest.importorskip("torch")
    assert torch.cuda.is_available(), "-m gpu run without a GPU"
    rng = np.random.default_rng(1000 * m + k)
    a = rng.standard_normal((m, k)) / np.sqrt(m)
    tau = np.array([2 / (1 + (a[i + 1:, i] ** 2).sum()) for i in range(k)])  # H_i orthogonal
    tau[::7] = 0.0                                                           # H_i = I
    c = rng.standard_normal((m, n))

    def dev(x, ld):
        buf = np.full((x.shape[1], ld), 7.25)
        buf[:, : x.shape[0]] = x.T
        return torch.tensor(buf, device="cuda")

    da, dc, dt = dev(a, m + pad), dev(c, m + pad), torch.tensor(tau, device="cuda")
    info = qrdm_amd.lib().qrdm_dormqr_dev(trans, m, n, k, da.data_ptr(), m + pad, dt.data_ptr(),
                                          dc.data_ptr(), m + pad, None)
    assert info == 0
    got = dc.cpu().numpy()
    assert (got[:, m:] == 7.25).all()
    assert (dt.cpu().numpy() == tau).all()
    want = apply_reflectors(a, tau, c, trans)
    # k orthogonal reflectors, each with an error of a few eps of the column's norm
    err = np.linalg.norm(got[:, :m].T - want.astype(float), axis=0)
    assert (err <= 8 * (k + 8) * 2.0 ** -53 * np.linalg.norm(c, axis=0)).all(), err.max()
