"""The next stage's input and the next leapfrog state, formed by the right-hand side's own
launch or by one behind it (large mixed systems): the same bits on either side of the sizes
where that changes, against the steps done one by one through the executor's calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def system(n, masses):
    import ode_prototyping_amd as oh
    x, m = oh.scenarios.plummer(n, seed=n)
    if masses == "spread":
        m = m * np.random.default_rng(n).uniform(0.5, 2.0, n)
    return x, None if masses == "unit" else m


# on 256 CUs the change comes at 8192 bodies with masses
@pytest.mark.parametrize("n,masses", [(4096, "equal"), (8192, "spread"), (8192, "equal"),
                                      (8193, "equal"), (8193, "spread"), (8193, "unit"),
                                      (16500, "spread")])
@pytest.mark.parametrize("tableau,fsal,near", [("DOPRI5", True, 0.0), ("DOP853", False, 0.0),
                                               ("DOPRI5", False, 20.0)])
def test_mixed_attempts(exe, n, masses, tableau, fsal, near):
    import ode_prototyping_amd as oh
    from ode_prototyping_amd.core import _Sub, tableau_shape
    x0, m = system(n, masses)
    ode = oh.NBodyODE(1e-2, m, "mixed")
    keep = exe.near_field
    try:
        exe.near_field = near
        res = oh.integrate(tableau, x0, 0.0, 10.0, 1e-10, 1e-10, ode, exe=exe, fsal=fsal,
                           max_accepted=3, trace_cap=32)
        x = oh.HipState(exe, data=x0)
        S = tableau_shape(tableau)[0]
        nv = x.size
        ks, y, out, err = (oh.HipState(exe, s * nv) for s in (S, 1, 1, 1))
        k = [_Sub(ks, j * nv, nv) for j in range(S)]
        for _, dt, accepted in res.trace:
            if not accepted:
                continue
            ode(exe, x, k[0])
            for stage in range(1, S):
                exe.rk_stage(tableau, stage, float(dt), y, ks, x)
                ode(exe, y, k[stage])
            exe.rk_update_state_and_error(tableau, float(dt), out, err, ks, x)
            x.assign(out)
        assert res.accepted == 3
        assert np.array_equal(bits(res.x_final), bits(x.to_numpy()))
    finally:
        exe.near_field = keep


@pytest.mark.parametrize("n,masses,near", [(8192, "spread", 0.0), (8193, "equal", 0.0),
                                           (8193, "unit", 0.0), (16384, "spread", 20.0),
                                           (16385, "equal", 20.0), (16385, "unit", 20.0)])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_mixed_leapfrog(exe, n, masses, near, steps):
    """Without output (one launch a step where the rule says so) and with it (three)."""
    import ode_prototyping_amd as oh
    x0, m = system(n, masses)
    ode = oh.NBodyODE(1e-2, m, "mixed")
    keep = exe.near_field
    try:
        exe.near_field = near
        tf = (steps - 0.5) * 1e-3
        out = oh.RawOutput()
        a, st = oh.leapfrog(x0, 0.0, tf, 1e-3, ode, exe=exe)
        b, _ = oh.leapfrog(x0, 0.0, tf, 1e-3, ode, out, exe=exe)
        assert st["steps"] == steps
        assert np.array_equal(bits(a), bits(b))
    finally:
        exe.near_field = keep
