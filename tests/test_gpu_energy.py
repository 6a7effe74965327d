"""Energies at the edges of the tile ring (one tile, an even and an odd number of tiles,
partial last tiles), without masses and without softening, against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from test_gpu_rhs import ic

pytestmark = pytest.mark.gpu


def energies(exe, x, n, eps, m):
    import ode_prototyping_amd as oh
    xs = oh.HipState(exe, data=x)
    ms = None if m is None else oh.HipState(exe, data=m)
    out = np.zeros(2)
    exe.check(oh.lib().odehip_nbody_energy(exe.handle, xs.ptr, n, eps, ms.ptr if ms else None,
                                           out.ctypes.data_as(C.POINTER(C.c_double))), "energy")
    return out


@pytest.mark.parametrize("n", [1, 2, 33, 64, 65, 128, 129, 192, 200, 1000, 4097])
@pytest.mark.parametrize("eps,masses", [(1e-3, True), (0.0, False)])
def test_energy_at_tile_edges(exe, n, eps, masses):
    x, m = ic(n, seed=n, masses=masses)
    ke, pe = O.energy(x, n, eps, m)
    got = energies(exe, x, n, eps, m)
    # every term to a few ulp, sums of one sign: far inside 1e-13
    assert abs(got[0] - ke) <= 1e-13 * abs(ke)
    assert abs(got[1] - pe) <= 1e-13 * abs(pe)


def test_energy_of_coincident_and_far_bodies(exe):
    """r = 0 without softening is infinitely bound; a square that overflows adds nothing."""
    x, m = ic(100, seed=5)
    y = x.copy()
    y[3 * 70:3 * 70 + 3] = y[:3]
    assert energies(exe, y, 100, 0.0, m)[1] == -np.inf
    y = x.copy()
    y[3 * 70] = 1e200
    pos = np.delete(x[:300].reshape(100, 3), 70, axis=0)
    keep = np.concatenate([pos.ravel(), np.zeros(297)])
    want = energies(exe, keep, 99, 1e-3, np.delete(m, 70))[1]
    got = energies(exe, y, 100, 1e-3, m)[1]
    assert abs(got - want) <= 1e-13 * abs(want)
