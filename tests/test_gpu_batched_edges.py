"""The batched form at the edges of its trailing update (32-row chunks of V and
C, 16-column groups, 128 columns a pass), its column moves (32-row blocks) and
its norms (four columns, groups of 256)."""
import numpy as np
import pytest

import inputs
from helpers import assert_parity
from test_gpu_batched import gpu, pack, run_batch, unpack  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(1, 1), (1, 3), (2, 70), (33, 17), (65, 66), (64, 81), (97, 82), (63, 193)],
    [(127, 129), (128, 192), (129, 208), (160, 321), (193, 65), (257, 340)],
    [(449, 193), (450, 209), (513, 130), (700, 90)],
])
def test_batched_edges(gpu, oracle, shapes):  # noqa: F811
    import qrdm_amd
    mats = [inputs.gaussian(m, n, 17 * m + n) * (1.0 + np.random.default_rng(m).permutation(n) / n)
            for m, n in shapes]
    plan = qrdm_amd.BatchPlan(shapes, nb=64)
    outs = run_batch(gpu, plan, pack(gpu, plan, mats))
    for i, a in enumerate(mats):
        print(shapes[i], flush=True)
        assert_parity(unpack(plan, i, *outs), oracle.dgeqrdm(a))
