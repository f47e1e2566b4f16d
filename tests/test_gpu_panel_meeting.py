"""Column-by-column panels of several workgroups: where their workgroups do not all
arrive (QRDM_PANEL=alone declines every one where they meet) the one-workgroup panel
gives the factors; and the limits between the forms of several workgroups and
the one-workgroup form that takes what is larger.  Reference: LAPACK's dgeqrf."""
import numpy as np
import pytest

from test_gpu_regpanel import check, gpu, lapack, qrf  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(449, 1), (449, 64), (600, 70), (4100, 65), (7000, 20)])
def test_declined_where_they_meet(gpu, monkeypatch, m, n):  # noqa: F811
    print("panel alone", m, n, flush=True)
    a = np.random.default_rng(m + n).standard_normal((m, n))
    monkeypatch.setenv("QRDM_PANEL", "alone")
    check(qrf(gpu, a), lapack(a))


@pytest.mark.parametrize("m,n", [(6272, 66), (6273, 66), (7000, 20), (28672, 8), (28673, 8)])
def test_forms_of_several_workgroups(gpu, m, n):  # noqa: F811
    print("panel form", m, n, flush=True)
    a = np.random.default_rng(m + n).standard_normal((m, n))
    check(qrf(gpu, a), lapack(a))


@pytest.mark.parametrize("scale", [0.0, 1e-170])
def test_range_above_6272_rows(gpu, scale):  # noqa: F811
    m, n = 6500, 12
    a = np.random.default_rng(5).standard_normal((m, n))
    a[:, 4] *= scale
    (g, t), (b, u) = qrf(gpu, a), lapack(a)
    keep = [c for c in range(n) if c != 4]
    assert np.linalg.norm((np.triu(g) - np.triu(b))[:, keep]) <= 1e-12 * np.linalg.norm(b)
    assert np.abs(t - u)[keep].max() <= 1e-12
    assert np.linalg.norm(np.triu(g)[:, 4] - np.triu(b)[:, 4]) <= 1e-12 * np.linalg.norm(a[:, 4])


@pytest.mark.parametrize("alone", [False, True])
@pytest.mark.parametrize("m,n", [(449, 1), (600, 70), (7000, 3)])
def test_every_column_fixed(gpu, monkeypatch, m, n, alone):  # noqa: F811
    import qrdm_amd
    if alone:
        monkeypatch.setenv("QRDM_PANEL", "alone")
    print("all fixed", m, n, alone, flush=True)
    a = np.random.default_rng(m * n).standard_normal((m, n))
    d = gpu.from_numpy(np.ascontiguousarray(a.T)).cuda()
    tau = gpu.zeros(n, dtype=gpu.float64, device="cuda")
    jp, nc = np.ones(n, np.int32), np.zeros(n, np.int32)
    info, _ = qrdm_amd.dgeqrdm_dev(d, m, tau, jp, nc, np.array([0.9, 0.15, 0.0]))
    assert info == 0 and np.array_equal(jp, np.arange(1, n + 1))
    check((d.cpu().numpy().T, tau.cpu().numpy()), lapack(a))
