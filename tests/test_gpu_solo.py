"""Solves by one workgroup per system against the lockstep rounds, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("variant,near,tableau,sizes", [
    # tile edges, whole and partial groups of 32 and chunks of 128 partners, the
    # largest sizes one workgroup takes (LDS at 12 and 13 stages) and the next
    ("exact", 0.0, "DOPRI5", [1, 2, 31, 32, 33, 64, 65, 96, 127, 128, 129]),
    ("exact", 0.0, "RKF78", [1, 63, 64, 65, 79, 80, 81, 82, 83, 84, 85, 100]),
    ("fast", 0.0, "DOP853", [1, 3, 33, 64, 127, 128, 129, 160, 192, 193, 200, 215, 222, 250]),
    ("fast", 0.0, "HE21", [65, 255, 256, 257]),
    ("mixed", 0.0, "RKF78", [2, 32, 95, 128, 129, 191, 192, 193, 200, 201, 202, 203, 204]),
    ("mixed", 20.0, "DOPRI5", [30, 64, 127, 129, 255, 256, 257])])
@pytest.mark.parametrize("controller", ["reference", "pi"])
def test_solo_equals_rounds(exe, variant, near, tableau, sizes, controller):
    """Equal, spread and unit masses, k1 reuse on and off; tile_config 7 keeps every
    system in the lockstep rounds."""
    import ode_prototyping_amd as oh
    from ode_prototyping_amd.ensemble import pack, solve_ensemble
    xs = [oh.scenarios.uniform_cube(n, seed=500 + n)[0] for n in sizes]
    rng = np.random.default_rng(9)
    spread = [rng.uniform(0.5, 2.0, n) / n if k % 2 else np.full(n, 1.0 / n)
              for k, n in enumerate(sizes)]
    exe.near_field = near
    try:
        for masses, fsal in ((pack(spread), False), (None, True)):
            runs = [solve_ensemble(tableau, sizes, pack(xs), 0.0, 1e-2, 1e-9, 1e-9, 1e-2, masses,
                                   variant=variant, exe=exe, fsal=fsal, controller=controller,
                                   trace_cap=256, tile_config=cfg, max_attempts=150)
                    for cfg in (-1, 7)]
            assert np.array_equal(runs[0].attempts, runs[1].attempts)
            assert np.array_equal(runs[0].rhs_evals, runs[1].rhs_evals)
            assert runs[0].status_names == runs[1].status_names
            assert np.array_equal(bits(runs[0].x_final), bits(runs[1].x_final))
            for a, b in zip(runs[0].trace, runs[1].trace):
                assert np.array_equal(bits(a), bits(b))
    finally:
        exe.near_field = oh.MIXED_NEAR_DEFAULT


@pytest.mark.parametrize("n", [2, 64, 128, 129])
def test_solo_single_solve_launch_boundaries(exe, n):
    """A solve of more attempts than one launch makes, k1 kept over the boundary, times
    and trace on, against the attempt-by-attempt launches."""
    import ode_prototyping_amd as oh
    x, m = oh.scenarios.uniform_cube(n, seed=n)
    runs = [oh.integrate("DOPRI5", x, 0.0, 5.0, 1e-10, 1e-10, oh.NBodyODE(1e-2, m, "exact"),
                         exe=exe, fsal=True, max_attempts=131, trace_cap=200,
                         attempts_per_launch=k) for k in (0, 5)]
    assert runs[0].accepted == runs[1].accepted and runs[0].rhs_evals == runs[1].rhs_evals
    assert np.array_equal(bits(runs[0].times), bits(runs[1].times))
    assert np.array_equal(bits(runs[0].trace), bits(runs[1].trace))
    assert np.array_equal(bits(runs[0].x_final), bits(runs[1].x_final))
