"""Rounding of the block updates against the stored reflectors applied in extended
precision.

C - V W is summed from zero and subtracted once: one rounding of each entry.
"""
import numpy as np
import pytest
import torch

import qrdm_amd

pytestmark = pytest.mark.gpu
LD = np.longdouble


def unit_lower(fac, k):
    v = np.tril(fac[:, :k], -1)
    v[np.arange(k), np.arange(k)] = 1.0
    return v


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
