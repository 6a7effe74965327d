"""Right-hand-side kernels at the edges of their shapes: sizes where the launcher changes
the targets per workgroup, partial chunks and tiles, the smallest and a size with several
rounds of workgroups; the exact variant bit for bit against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_rhs import gpu_rhs, ic

pytestmark = pytest.mark.gpu

EDGES = [1, 16, 64, 65, 255, 256, 257, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4111, 4353,
         8177, 8705]


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("form", ["unit", "masses", "ieee"])
def test_exact_rhs_at_shape_edges(exe, n, form):
    x, m = ic(n, seed=n + 1, masses=form != "unit")
    if form == "masses":
        m = m * (1.0 + 0.5 * np.random.default_rng(n).random(n))
    eps = 1e-3
    if form == "ieee":  # a coordinate below 2^-246 sends every term to the IEEE expressions
        x[3 * (n - 1)] = 1e-80
    got = gpu_rhs(exe, x, eps, m, "exact")
    want = O.rhs(O.RHS_NBODY, x, eps, m, threads=8)
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64)), \
        f"n={n}: max abs diff {np.max(np.abs(got - want))}"


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256, 257, 512, 513, 517, 1027, 11467, 11521])
@pytest.mark.parametrize("eps,masses", [(1e-2, False), (1e-2, True), (0.0, True)])
def test_fast_rhs_at_shape_edges(exe, n, eps, masses):
    x, m = ic(n, seed=n + 2, masses=masses)
    got = gpu_rhs(exe, x, eps, m, "fast")
    want = O.rhs(O.RHS_NBODY, x, eps, m, threads=8)
    assert np.array_equal(got[:3 * n], want[:3 * n])
    scale = np.max(np.abs(want[3 * n:])) if n > 1 else 1.0
    assert np.max(np.abs(got - want)) <= 5e-14 * scale  # the variant's bar


@pytest.mark.parametrize("n", [33000, 40000])
def test_exact_rhs_several_workgroups_per_cu(exe, n):
    """Two and more 64-target workgroups per CU (four waves each); rows of a few targets
    against the oracle's order: the sums over the partners one by one."""
    x, m = ic(n, seed=n, masses=True)
    got = gpu_rhs(exe, x, 1e-3, m, "exact")
    p = x[:3 * n].reshape(n, 3)
    assert np.array_equal(got[:3 * n], x[3 * n:])
    for i in (0, 63, 64, n // 2, n - 1):
        d = p - p[i]
        s = ((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]) + 1e-3 * 1e-3
        den = np.sqrt(s) * s
        t = d / den[:, None] * m[:, None]
        t[i] = 0.0
        want = np.cumsum(t, axis=0)[-1]  # in partner order
        assert np.array_equal(got[3 * n + 3 * i:3 * n + 3 * i + 3], want)
