"""Finite inputs whose updates overflow: some partial norms become NaN.  The call ends,
with every column in jpvt once (a NaN among the sort's keys must not lose or invent
an index)."""
import numpy as np
import pytest

from test_gpu_regpanel import gpu  # noqa: F401

pytestmark = pytest.mark.gpu


def near_overflow(m, n):
    """Column norms just below the largest double, each column twice: tau (V^T C)
    overflows where tau > 1.01."""
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n // 2))
    a = np.hstack([a, a])
    return a / np.linalg.norm(a, axis=0) * 1.78e308


@pytest.mark.parametrize("m,n,nb", [(100, 160, 80), (300, 1200, 128), (100, 160, 64), (300, 1200, 32)])
def test_steps(gpu, m, n, nb):  # noqa: F811
    import qrdm_amd
    print("overflow", m, n, nb, flush=True)
    d = gpu.from_numpy(np.ascontiguousarray(near_overflow(m, n).T)).cuda()
    tau = gpu.zeros(min(m, n), dtype=gpu.float64, device="cuda")
    jp, nc = np.zeros(n, np.int32), np.zeros(n, np.int32)
    info, _ = qrdm_amd.dgeqrdm_dev(d, m, tau, jp, nc, np.array([0.9, 0.15, 0.0]), nb=nb)
    assert info == 0
    assert not bool(gpu.isfinite(d).all())  # the case is what it says
    assert np.array_equal(np.sort(jp), np.arange(1, n + 1))


@pytest.mark.parametrize("rows", [0, 128])
def test_batched(gpu, rows):  # noqa: F811
    import qrdm_amd
    shapes = [(100, 160), (300, 280)]
    plan = qrdm_amd.BatchPlan(shapes, nb=64)
    plan.set_panel_rows(rows)
    buf = gpu.from_numpy(np.concatenate([near_overflow(m, n).T.ravel() for m, n in shapes])).cuda()
    tau = gpu.zeros(380, dtype=gpu.float64, device="cuda")
    jp, nc, info = (gpu.zeros(q, dtype=gpu.int32, device="cuda") for q in (440, 440, 2))
    plan.run(buf, tau, jp, nc, info, thres=(0.9, 0.15, 0.0), stop=0, graph=False)
    gpu.cuda.synchronize()
    jp = jp.cpu().numpy()
    assert not bool(gpu.isfinite(buf).all())
    assert np.array_equal(np.sort(jp[:160]), np.arange(1, 161))
    assert np.array_equal(np.sort(jp[160:]), np.arange(1, 281))
