"""Batched fast and mixed right-hand sides whose tiles are shared by several waves, on either
side of the sizes at which such a launch takes 16-target workgroups (128 tiles, 1024 bodies):
bit for bit the sums of one wave per tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("sizes", [
    [1], [16, 17, 33], [1024], [1, 15, 16, 31, 32, 33, 63, 64, 65, 128, 129, 255, 257, 1000, 1023],
    [1025], [64] * 127, [64] * 128, [64] * 128 + [3], [1024] * 8, [1000] * 8 + [5]],
    ids=lambda s: f"{len(s)}x{max(s)}")
@pytest.mark.parametrize("variant", ["fast", "mixed"])
@pytest.mark.parametrize("masses,eps", [("equal", 1e-3), ("spread", 1e-3), ("unit", 0.0)])
def test_shared_tiles(exe, sizes, variant, masses, eps):
    import ode_prototyping_amd as oh
    from ode_prototyping_amd.ensemble import ensemble_rhs, pack
    cubes = [oh.scenarios.uniform_cube(n, seed=31 + k) for k, n in enumerate(sizes)]
    x, m = pack(c[0] for c in cubes), pack(c[1] for c in cubes)
    if masses == "spread":
        m = m * np.random.default_rng(len(sizes)).uniform(0.5, 2.0, m.size)
    keep = exe.near_field
    try:
        exe.near_field = 0.0
        run = [ensemble_rhs(exe, sizes, x, eps, None if masses == "unit" else m, variant,
                            tile_config=cfg)[0] for cfg in (6, 12, 13, 14, 15, 16, 17)]
    finally:
        exe.near_field = keep
    for got in run[1:]:
        assert np.array_equal(bits(got), bits(run[0]))
