"""The register-held column-by-column panel at the edges of its forms.

The unpivoted QR runs it on every panel: one workgroup of four waves up to
128 rows, of seven up to 336 and 448, several workgroups above; a panel
whose sums of squares leave the safe range is declined and taken by the
memory-based form.  Reference: LAPACK's dgeqrf (scipy).  Bar: R normwise and
the reflectors within 64 m eps cond-free for Gaussian input, 1e-12 here.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qrdm_amd
    qrdm_amd.lib()
    return torch


def qrf(torch, a, lda=None):
    import qrdm_amd
    m, n = a.shape
    lda = lda or m
    buf = np.full((n, lda), 7.25)
    buf[:, :m] = a.T
    d = torch.from_numpy(buf).cuda()
    tau = torch.zeros(min(m, n), dtype=torch.float64, device="cuda")
    info = qrdm_amd.lib().qrdm_dgeqrf_dev(m, n, d.data_ptr(), lda, tau.data_ptr(), None)
    assert info == 0, (info, qrdm_amd.last_error())
    out = d.cpu().numpy()
    assert np.all(out[:, m:] == 7.25)  # rows past m untouched
    return out[:, :m].T, tau.cpu().numpy()


def lapack(a):
    from scipy.linalg import lapack as ll
    qr, tau, _, info = ll.dgeqrf(np.asfortranarray(a))
    assert info == 0
    return qr, tau


def check(got, ref, tol=1e-12):
    (a, t), (b, u) = got, ref
    assert np.linalg.norm(np.triu(a) - np.triu(b)) <= tol * np.linalg.norm(np.triu(b))
    assert np.abs(np.tril(a, -1) - np.tril(b, -1)).max() <= tol
    assert np.abs(t - u).max() <= tol


@pytest.mark.parametrize("m,n,pad", [
    (1, 1, 0), (2, 2, 1), (15, 15, 0), (33, 16, 3), (64, 64, 0), (127, 70, 0), (128, 128, 0),
    (129, 17, 0), (192, 300, 5), (336, 64, 0), (337, 65, 0), (448, 100, 0), (449, 64, 0),
    (896, 40, 0), (897, 130, 7), (4100, 65, 0), (40, 90, 0)])
def test_sizes(gpu, m, n, pad):
    print("regpanel", m, n, pad, flush=True)
    a = np.random.default_rng(100 * m + n).standard_normal((m, n))
    check(qrf(gpu, a, m + pad), lapack(a))


@pytest.mark.parametrize("m", [100, 300, 1500])
@pytest.mark.parametrize("kind", ["triangular", "zerocols", "tiny", "huge", "mixed"])
def test_range(gpu, m, kind):
    """Columns with nothing below the diagonal (tau = 0), zero columns, and
    scales whose squares underflow or overflow (declined panels)."""
    print("regpanel range", m, kind, flush=True)
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, 80))
    if kind == "triangular":
        a = np.triu(a)
    elif kind == "zerocols":
        a[:, 3:9] = 0.0
        a[:, 70] = 0.0
    elif kind == "tiny":
        a *= 1e-170
    elif kind == "huge":
        a *= 1e160
    else:
        a[:, 10] *= 1e-200
        a[:, 40] *= 1e-180
    (g, t), (b, u) = qrf(gpu, a), lapack(a)
    scale = np.abs(b).max()
    if kind in ("tiny", "huge"):
        check((g / scale, t), (b / scale, u), 1e-11)
        return
    # column by column: R within 1e-12 of its column's norm
    nr = np.linalg.norm(a, axis=0)
    if kind in ("triangular", "zerocols"):
        assert np.all(np.linalg.norm(np.triu(g) - np.triu(b), axis=0) <= 1e-12 * np.maximum(nr, 1))
        if kind == "triangular":
            assert np.array_equal(g, a) and not t.any()
    else:
        # H_79 .. H_0 a = R column by column, each column to its own scale
        assert np.all(np.isfinite(g)) and np.all((t == 0) | ((t >= 1) & (t <= 2)))
        keep = [c for c in range(80) if c not in (10, 40)]
        d = np.linalg.norm(np.triu(g) - np.triu(b), axis=0)[keep]
        assert np.all(d <= 1e-12 * nr[keep])


def test_nan_stays_in_its_columns(gpu):
    """A NaN makes the panel's sums NaN: the memory-based form takes it and
    the call ends (LAPACK's dgeqrf gives NaN from that column on as well)."""
    a = np.random.default_rng(5).standard_normal((200, 70))
    a[150, 20] = np.nan
    g, t = qrf(gpu, a)
    b, u = lapack(a)
    lead = slice(0, 20)
    assert np.abs(np.triu(g)[:20, lead] - np.triu(b)[:20, lead]).max() <= 1e-12
    assert np.isnan(g[:, 20]).any()


@pytest.mark.parametrize("m,n,nb", [(600, 300, 96), (1400, 200, 130), (300, 280, 256)])
def test_wide_blocks(gpu, m, n, nb):
    """A DM block wider than 64 columns is reduced in parts: pivots and R
    against the oracle, with a truncation that ends in a later part."""
    import sys
    import os
    sys.path.insert(0, os.path.join(os.path.dirname(__file__), "golden"))
    import inputs
    from oracle import pyoracle as po
    import qrdm_amd
    for a in (inputs.gaussian(m, n, m), inputs.lowrank_noise(m, n, 90, n, noise=1e-7)):
        print("regpanel wide", m, n, nb, flush=True)
        ref = po.dgeqrdm(a, nb=nb, stop=3, eta=1e-5)
        d = gpu.from_numpy(np.ascontiguousarray(a.T)).cuda()
        tau = gpu.zeros(min(m, n), dtype=gpu.float64, device="cuda")
        jp, nc = np.zeros(n, np.int32), np.zeros(n, np.int32)
        nc[0] = 3
        info, _ = qrdm_amd.dgeqrdm_dev(d, m, tau, jp, nc, np.array([0.9, 0.15, 1e-5]), nb=nb)
        assert info == 0
        assert np.array_equal(jp, ref["jpvt"])
        assert np.array_equal(nc[:len(ref["ncols"])], ref["ncols"])
        R, Rr = np.triu(d.cpu().numpy().T), np.triu(ref["a"])
        assert np.linalg.norm(R - Rr) <= 1e-12 * np.linalg.norm(Rr)
