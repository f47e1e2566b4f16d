"""Rounding of the block updates: W = T^T V^T C and C - V W against the stored
reflectors applied in extended precision.

V^T C is a sum over all rows, so its error grows with the length of the longest
sum taken in one piece.  The bound is the error of a plain float64 emulation
with sixteen row slabs (four for the batched form, whose workgroup has four
waves), each summed in one piece, everything else exact.  C - V W is summed from
zero and subtracted once: one rounding of each entry.
"""
import ctypes

import numpy as np
import pytest
import torch

import qrdm_amd

pytestmark = pytest.mark.gpu
LD = np.longdouble
TH = np.array([0.9, 0.15, 0.0])


def vp(t):
    return ctypes.c_void_p(t.data_ptr())


def gaussian(m, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(n, m, generator=g, device="cuda", dtype=torch.float64)


def unit_lower(fac, k):
    v = np.tril(fac[:, :k], -1)
    v[np.arange(k), np.arange(k)] = 1.0
    return v


def wy_t(v, tau):
    """T of H_1 ... H_k = I - V T V^T, in extended precision."""
    k = tau.size
    s = v.astype(LD).T @ v.astype(LD)
    t = np.zeros((k, k), LD)
    for i in range(k):
        t[:i, i] = -tau[i] * (t[:i, :i] @ s[:i, i])
        t[i, i] = tau[i]
    return t


def sums_in_slabs(v, c, slabs):
    """V^T C with each slab's rows summed one after the other in float64."""
    edges = np.linspace(0, v.shape[0], slabs + 1).astype(int)
    p = np.zeros((v.shape[1], c.shape[1]))
    for a, b in zip(edges[:-1], edges[1:]):
        acc = np.zeros_like(p)
        for r in range(a, b):
            acc += np.outer(v[r], c[r])
        p += acc
    return p


def check_block(got, c, v, tau, trans, slabs, rows):
    """got: the first rows of (I - V op(T) V^T) C as the library computed them."""
    t = wy_t(v, tau)
    t = t.T if trans else t
    top = v[:rows].astype(LD)
    exact = c[:rows] - top @ (t @ (v.astype(LD).T @ c.astype(LD)))
    emul = c[:rows] - top @ (t @ sums_in_slabs(v, c, slabs).astype(LD))
    err = np.linalg.norm((got[:rows] - exact).astype(float))
    bound = np.linalg.norm((emul - exact).astype(float))
    assert err <= bound, (err, bound, err / bound)


def some_columns(lo, n):
    return np.linspace(lo, n - 1, 8).astype(int)


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("m,n", [(8192, 8192), (3001, 8191)])
def test_ormqr_block(m, n, trans):
    k = 64
    a = gaussian(m, k, 1)
    tau = torch.zeros(k, dtype=torch.float64, device="cuda")
    assert qrdm_amd.lib().qrdm_dgeqrf_dev(m, k, vp(a), m, vp(tau), None) == 0
    c = gaussian(m, n, 2)
    cols = some_columns(0, n)
    c0 = c[cols].cpu().numpy().T
    assert qrdm_amd.lib().qrdm_dormqr_dev(trans, m, n, k, vp(a), m, vp(tau), vp(c), m, None) == 0
    check_block(c[cols].cpu().numpy().T, c0, unit_lower(a.cpu().numpy().T, k),
                tau.cpu().numpy(), trans, 16, m)


def test_geqrf_first_block():
    m, n, k = 4096, 8192, 64
    a = gaussian(m, n, 3)
    cols = some_columns(k, n)
    c0 = a[cols].cpu().numpy().T
    tau = torch.zeros(m, dtype=torch.float64, device="cuda")
    assert qrdm_amd.lib().qrdm_dgeqrf_dev(m, n, vp(a), m, vp(tau), None) == 0
    fac = a[:k].cpu().numpy().T
    check_block(a[cols].cpu().numpy().T, c0, unit_lower(fac, k), tau[:k].cpu().numpy(), 1, 16, k)


@pytest.mark.parametrize("m,n,nb", [(8192, 8192, 64), (2048, 8000, 128)])
def test_dm_first_step(m, n, nb):
    a = gaussian(m, n, 4)
    a0 = a.clone()
    tau = torch.zeros(min(m, n), dtype=torch.float64, device="cuda")
    jp, nc = np.zeros(n, np.int32), np.zeros(n, np.int32)
    info, _ = qrdm_amd.dgeqrdm_dev(a, m, tau, jp, nc, TH, nb=nb)
    assert info == 0
    k = min(int(nc[0]), 64)
    cols = some_columns(n // 2, n)
    c0 = a0[torch.from_numpy(jp[cols].astype(np.int64) - 1).cuda()].cpu().numpy().T
    fac = a[:k].cpu().numpy().T
    check_block(a[cols].cpu().numpy().T, c0, unit_lower(fac, k), tau[:k].cpu().numpy(), 1, 16, k)


def test_batched_first_step():
    m, n = 1024, 512
    it = (qrdm_amd.BatchItem * 1)(qrdm_amd.BatchItem(m, n, m, 0, 0, 0, 0))
    lib = qrdm_amd.lib()
    plan = lib.qrdm_batch_plan_create(1, it, 64)
    assert plan
    a = gaussian(m, n, 5)
    a0 = a.clone()
    tau = torch.zeros(n, dtype=torch.float64, device="cuda")
    jp, nc, info = (torch.zeros(q, dtype=torch.int32, device="cuda") for q in (n, n, 1))
    assert lib.qrdm_dgeqrdm_batched(plan, vp(a), vp(tau), vp(jp), vp(nc), vp(info),
                                    TH.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 0, 0,
                                    None) == 0
    torch.cuda.synchronize()
    lib.qrdm_batch_plan_destroy(plan)
    assert int(info[0]) == 0
    k = int(nc[0])
    cols = np.arange(n // 2, n, 8)
    c0 = a0[(jp.long() - 1)[torch.from_numpy(cols).cuda()]].cpu().numpy().T
    fac = a[:k].cpu().numpy().T
    check_block(a[cols].cpu().numpy().T, c0, unit_lower(fac, k), tau[:k].cpu().numpy(), 1, 4, k)


@pytest.mark.parametrize("left", [1e-5, 1e-2])
def test_update_rounds_each_entry_once(left):
    # C is the panel's columns combined, and entries of size left / 16 on the lower
    # rows, where V is so small that V W changes them by a thousandth: one rounding of
    # the result, and 64 of V W, 64 / 2 / 1000 of one.  left = 1e-5 recomputes the
    # columns' norms (and updates them then), 1e-2 downdates them.
    m, q, low = 512, 40, 256
    rng = np.random.default_rng(6)
    panel = rng.standard_normal((m, 64))
    panel[low:] *= 1e-4 * left
    c = panel @ (rng.standard_normal((64, q)) / 64)
    c[low:] += rng.standard_normal((m - low, q)) * left / 16
    a0 = np.hstack([panel, c])
    a = torch.from_numpy(np.ascontiguousarray(a0.T)).cuda()
    n = 64 + q
    tau = torch.zeros(n, dtype=torch.float64, device="cuda")
    jp, nc = np.zeros(n, np.int32), np.zeros(n, np.int32)
    nc[0] = 3  # stop once the remaining block's bound is below half the largest norm
    info, _ = qrdm_amd.dgeqrdm_dev(a, m, tau, jp, nc, np.array([0.9, 0.15, 0.5]), nb=64)
    assert info == 0 and nc[0] == 64 and nc[1] == 0 and jp[:64].max() == 64
    fac = a.cpu().numpy().T
    x = a0[:, jp - 1].astype(LD)[:, 64:]
    t = tau.cpu().numpy()
    for i in range(64):
        v = unit_lower(fac, 64)[:, i].astype(LD)
        x -= np.outer(t[i] * v, v @ x)
    got = fac[low:, 64:]
    err = np.abs((got - x[low:]).astype(float))
    assert (err <= 0.5 * np.spacing(np.abs(got)) + 0.1 * np.spacing(left / 16)).all()
