"""Leapfrog without output (one launch a step, the update in the right-hand side's
epilogue) bit for bit against the oracle, in every shape of the exact kernels: one, two,
four and eight targets a workgroup, 16 and 32 with an overlapping last workgroup, 64."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("n,steps", [(1, 3), (64, 1), (64, 2), (64, 51), (300, 3), (300, 4),
                                     (513, 2), (1000, 3), (1025, 2), (2047, 3), (2049, 2),
                                     (4111, 3), (8177, 2), (8705, 2), (16385, 1)])
@pytest.mark.parametrize("masses", [False, True])
def test_exact(exe, n, steps, masses):
    import ode_prototyping_amd as oh
    x, m = oh.scenarios.uniform_cube(n, seed=n)
    m = m * np.random.default_rng(n).uniform(0.5, 2.0, n) if masses else None
    tf = (steps - 0.5) * 1e-3
    ode = oh.NBodyODE(1e-3, m, "exact")
    xf, st = oh.leapfrog(x, 0.0, tf, 1e-3, ode, exe=exe)
    ref = O.leapfrog(x, 0.0, tf, 1e-3, softening=1e-3, masses=m, store_states=False, threads=8)
    assert st["steps"] == ref.accepted == steps
    assert np.array_equal(bits(xf), bits(ref.x_final))


@pytest.mark.parametrize("variant,near", [("fast", 0.0), ("mixed", 0.0), ("mixed", 20.0)])
@pytest.mark.parametrize("n,steps", [(65, 2), (255, 3), (1027, 3), (11500, 2), (17000, 1)])
def test_reorderable(exe, variant, near, n, steps):
    """... and the other variants against their runs that keep every state (three launches
    a step with the same right-hand sides)."""
    import ode_prototyping_amd as oh
    x, m = oh.scenarios.plummer(n, seed=n)
    ode = oh.NBodyODE(1e-2, m * np.random.default_rng(n).uniform(0.5, 2.0, n), variant)
    keep = exe.near_field
    try:
        exe.near_field = near
        tf = (steps - 0.5) * 1e-3
        a, _ = oh.leapfrog(x, 0.0, tf, 1e-3, ode, exe=exe)
        b, st = oh.leapfrog(x, 0.0, tf, 1e-3, ode, oh.RawOutput(), exe=exe)
        assert st["steps"] == steps
        assert np.array_equal(bits(a), bits(b))
    finally:
        exe.near_field = keep
