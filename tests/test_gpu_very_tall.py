"""More rows than 32-bit byte offsets over sixteen columns of V can reach, in a process
of its own (its workspace is 73 GB)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import ctypes
import torch
import qrdm_amd
m, k = 36_000_000, 16
g = torch.Generator(device="cuda").manual_seed(1)
a = torch.randn(k, m, generator=g, device="cuda", dtype=torch.float64) * m ** -0.5
c = torch.randn(1, m, generator=g, device="cuda", dtype=torch.float64)
tau = torch.empty(k, dtype=torch.float64, device="cuda")
want = c.clone()
for i in range(k):  # Q^T c, a reflector after the other
    v = a[i].clone()
    v[:i] = 0
    v[i] = 1
    tau[i] = 2 / v.dot(v)
    want[0] -= tau[i] * v.dot(want[0]) * v
p = lambda t: ctypes.c_void_p(t.data_ptr())
assert qrdm_amd.lib().qrdm_dormqr_dev(1, m, 1, k, p(a), m, p(tau), p(c), m, None) == 0
print("error", ((c - want).norm() / want.norm()).item())
"""


@pytest.mark.gpu
def test_ormqr_36_million_rows():
    print("ormqr 36000000 x 1, 16 reflectors", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    err = float(r.stdout.split("error")[1])
    assert err <= 1e-14, err
