"""Attempts enqueued behind a solve's last one do no dense-output work: the last step's
pass runs once, whether or not that step covers an output time.

A replay holds far more attempts than the solve makes, so the passes that a last step with
its gate left open would repeat -- one for each surplus attempt of the first replay at least,
four right-hand sides each -- cost several times what they may.  Both solves of a comparison
make the same attempts and one dense pass each."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ATTEMPTS = 48  # enqueued per replay


def best(f, reps=8):
    f()
    t = []
    for _ in range(reps):
        a = time.perf_counter()
        f()
        t.append(time.perf_counter() - a)
    return min(t)


def rhs_seconds(exe, ode, x):
    import ode_prototyping_amd as oh
    xs, ks = oh.HipState(exe, data=x), oh.HipState(exe, data=x)
    exe.timer_start()
    for _ in range(20):
        ode(exe, xs, ks)
    return exe.timer_stop() / 20 * 1e-3


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("fsal", [False, True])
def test_single_solve(exe, fsal):
    import ode_prototyping_amd as oh
    n, steps = 6000, 4
    x, m = oh.scenarios.plummer(n, seed=3)
    ode = oh.NBodyODE(1e-2, m, "exact")

    def solve(dense):
        return oh.integrate("DOP853", x, 0.0, 10.0, 1e-10, 1e-10, ode, exe=exe, fsal=fsal,
                            max_accepted=steps, attempts_per_launch=ATTEMPTS, dense_times=dense)
    t = solve(None).times
    early, late = [0.5 * (t[1] + t[2])], [0.5 * (t[-2] + t[-1])]
    a, b = solve(early), solve(late)
    assert a.n_dense == b.n_dense == 1 and a.dense_steps == b.dense_steps == 1
    assert a.attempts == b.attempts < ATTEMPTS // 2
    assert np.array_equal(bits(a.x_final), bits(b.x_final))
    repeated = ATTEMPTS // 2 * 4 * rhs_seconds(exe, ode, x)
    assert best(lambda: solve(late)) - best(lambda: solve(early)) < repeated / 4


def test_ensemble(exe):
    import ode_prototyping_amd as oh
    from ode_prototyping_amd.ensemble import pack, solve_ensemble
    # the same system four times: one output time inside everyone's last step
    sizes = [3000] * 4
    x, m = (pack([v] * 4) for v in oh.scenarios.plummer(3000, seed=7))
    one = oh.NBodyODE(1e-2, None, "fast")

    def solve(dense):
        return solve_ensemble("DOP853", sizes, x, 0.0, 10.0, 1e-10, 1e-10, 1e-2, m,
                              variant="fast", exe=exe, max_accepted=4, trace_cap=64,
                              rounds_per_launch=ATTEMPTS, dense_times=dense)
    rows = solve(None).trace[0]
    t = np.cumsum(rows[rows[:, 2] == 1.0, 1])
    early, late = [0.5 * (t[0] + t[1])], [0.5 * (t[-2] + t[-1])]
    a, b = solve(early), solve(late)
    assert np.all(a.n_dense == 1) and np.all(b.n_dense == 1)
    assert np.array_equal(a.attempts, b.attempts) and max(a.attempts) < ATTEMPTS // 2
    assert np.array_equal(bits(a.x_final), bits(b.x_final))
    repeated = ATTEMPTS // 2 * 4 * rhs_seconds(exe, one, x[:6 * sizes[0]])
    assert best(lambda: solve(late)) - best(lambda: solve(early)) < repeated / 4
