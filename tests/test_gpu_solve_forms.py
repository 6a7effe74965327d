"""A solve's bits do not depend on what output is asked for or on how its attempts are
launched: the one-workgroup form of small systems (no output but times and trace, default
launches) against graph replays, direct launches, kept states and dense output."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def same(a, b):
    assert (a.accepted, a.rejected, a.status) == (b.accepted, b.rejected, b.status)
    assert np.array_equal(bits(a.times), bits(b.times))
    assert np.array_equal(bits(a.trace), bits(b.trace))
    assert np.array_equal(bits(a.x_final), bits(b.x_final))


# levels of the 64-lane fold that lack lanes, one and several tiles and sets, the largest
# sizes of the form (HE21: by its rule, DOP853: by LDS) and the next
@pytest.mark.parametrize("variant,tableau,sizes", [
    ("fast", "DOPRI5", [1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65]),
    ("fast", "DOP853", [40, 66, 127, 128, 129, 191, 192, 193, 200, 201, 202, 203]),
    ("fast", "HE21", [100, 160, 255, 256, 257]),
    ("exact", "DOPRI5", [5, 64, 65, 127, 128, 129]),
    ("exact", "DOP853", [33, 95, 128])])
@pytest.mark.parametrize("masses,eps", [("unit", 1e-2), ("equal", 1e-2), ("spread", 1e-2),
                                        ("spread", 0.0), ("unit", 0.0)])
def test_forms_agree(exe, variant, tableau, sizes, masses, eps):
    import ode_prototyping_amd as oh
    for n in sizes:
        x, m = oh.scenarios.uniform_cube(n, seed=900 + n)
        if masses == "spread":
            m = m * np.random.default_rng(n).uniform(0.5, 2.0, n)
        ode = oh.NBodyODE(eps, None if masses == "unit" else m, variant)
        fsal = n % 2 == 0

        def solve(**kw):
            return oh.integrate(tableau, x, 0.0, 1e-2, 1e-11, 1e-11, ode, exe=exe, fsal=fsal,
                                max_attempts=40, trace_cap=64, **kw)
        print(f"{variant} {tableau} n={n} {masses} eps={eps}", flush=True)
        plain = solve()
        same(plain, solve(attempts_per_launch=7))
        same(plain, solve(attempts_per_launch=-1))
        out = oh.RawOutput()
        kept = solve(output=out)
        same(plain, kept)
        assert np.array_equal(bits(out.states()[-1]), bits(plain.x_final))
        if tableau in ("DOPRI5", "DOP853") and len(plain.times) > 2:
            times = [0.5 * (plain.times[1] + plain.times[2])]
            dense = solve(dense_times=times)
            assert dense.n_dense == 1
            if tableau == "DOPRI5" or not fsal:  # (DOP853's pass gives k1 with reuse on)
                same(plain, dense)


@pytest.mark.parametrize("controller", ["pi", "learned"])
def test_fast_forms_agree_with_other_controllers(exe, controller):
    import ode_prototyping_amd as oh
    from ode_prototyping_amd import train_controller as trc
    net = trc.pretrained(exe, "DOP853", "fast")[0] if controller == "learned" else None
    for n in (24, 64, 130, 180):
        x, m = oh.scenarios.plummer(n, seed=n)
        ode = oh.NBodyODE(1e-2, m, "fast")
        runs = [oh.integrate("DOP853", x, 0.0, 0.3, 1e-10, 1e-10, ode, exe=exe, max_attempts=90,
                             trace_cap=128, controller=controller, mlp=net,
                             attempts_per_launch=k) for k in (0, 5)]
        same(*runs)
