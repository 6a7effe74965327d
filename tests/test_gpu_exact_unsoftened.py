"""Exact right-hand side without softening (IEEE square root and divisions throughout, in
instances of their own) bit for bit against the oracle: whole and partial chunks of the 16- and
32-target kernels, their overlapping last workgroup, and the shapes on either side."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_rhs import gpu_rhs, ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7, 300, 1025, 2048, 2049, 2064, 2065, 3119, 4096, 4097, 4104,
                               4105, 8183, 8192, 8193, 16393])
@pytest.mark.parametrize("masses", [False, True])
def test_unsoftened(exe, n, masses):
    x, m = ic(n, seed=n + 5, masses=masses)
    if masses:
        m = m * (1.0 + 0.5 * np.random.default_rng(n).random(n))
    got = gpu_rhs(exe, x, 0.0, m, "exact")
    want = O.rhs(O.RHS_NBODY, x, 0.0, m, threads=8)
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
