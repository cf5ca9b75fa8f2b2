"""Ray queries at the limits of their input: rays that cannot hit anything (a range that is not
positive or NaN, an origin that is not finite or so far away that every box distance overflows) among
ordinary rays of the same waves. They report misses; the CPU BVH (oracle/pt_oracle.cpp, box_hit) rejects
them at its root.
"""
import numpy as np
import pytest

import prender_amd as pa
import raygen

pytestmark = pytest.mark.gpu

NAN, INF = np.nan, np.inf


def words(hits):
    return hits.view(np.uint32)


DOWN, UP = (-0.6, -0.64, -0.48), (0.6, 0.64, 0.48)
# (origin, direction, tMax)
HOPELESS = [
    ((NAN, NAN, NAN), DOWN, INF), ((NAN, NAN, NAN), UP, 10), ((NAN, 0, 0), DOWN, INF), ((0, NAN, 0), UP, INF),
    ((0, 0, NAN), (0, 0, 1), INF), ((INF, INF, INF), DOWN, INF), ((-INF, -INF, -INF), UP, INF), ((INF, 0, 0), DOWN, INF),
    ((0, 0.5, -INF), (0, 0, 1), INF), ((3e38, 3e38, 3e38), DOWN, INF), ((3e38, 3e38, 3e38), DOWN, 3.4028235e38),
    ((0, 0.5, 0), UP, NAN), ((0, 0.5, 0), DOWN, 0), ((0, 0.5, 0), UP, -1), ((0, 0.5, 0), DOWN, -INF),
]


@pytest.mark.parametrize("n", [len(HOPELESS), 1003, 200003])
def test_rays_that_hit_nothing_among_others(plugin, c1, n):
    lo, hi = raygen.scene_bounds(c1)
    rays = raygen.random_rays(lo, hi, n, 5)
    good = np.random.default_rng(n).random(n) < 0.5
    want = np.zeros(n, pa.HIT_DTYPE)
    want["prim"] = -1
    occluded = np.zeros(n, bool)
    want[good] = plugin.trace(c1, rays[good])
    occluded[good] = plugin.trace(c1, rays[good], any_hit=True)["prim"] >= 0
    for i in np.flatnonzero(~good):
        rays["o"][i], rays["d"][i], rays["tMax"][i] = HOPELESS[i % len(HOPELESS)]
    got = plugin.trace(c1, rays)
    assert np.array_equal(words(got), words(want))
    assert np.array_equal(plugin.trace(c1, rays, any_hit=True)["prim"] >= 0, occluded)
