"""Wide steps at the edges of their kernels: sort lists of 1024 keys, candidate
tiles of 64, row slabs of the Gram, batches of 16 swaps that share columns."""
import numpy as np
import pytest

import inputs
from helpers import assert_parity
from test_gpu_wide import gpu, run_host  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,nb,delta,tau", [
    (70, 66, 65, 0.9, 0.15),      # one row slab and a bit, two candidate tiles
    (140, 2500, 100, 0.9, 0.15),  # three sort lists, two passes
    (4100, 260, 256, 0.9, 0.15),  # many slabs, ten tile pairs
    (700, 500, 128, 0.08, 0.0),   # few accepted: the accepted columns far apart
    (700, 500, 192, 0.9, 0.999),  # a handful of candidates
])
def test_wide_edges(gpu, oracle, m, n, nb, delta, tau):  # noqa: F811
    a = inputs.gaussian(m, n, m + nb)
    a *= 1.0 + np.random.default_rng(nb).permutation(n) / n  # spread norms: real moves
    got = run_host(a, nb=nb, delta=delta, tau=tau)
    ref = oracle.dgeqrdm(a, nb=nb, delta=delta, tau=tau)
    assert_parity(got, ref, strict=True)
