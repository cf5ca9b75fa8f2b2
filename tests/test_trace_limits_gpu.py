"""Ray queries at the limits of their input: rays that cannot hit anything (a range that is not
positive or NaN, an origin that is not finite or so far away that every box distance overflows) among
ordinary rays of the same waves, and ranges that end one float above the hit.

The former report misses, as the CPU BVH (oracle/pt_oracle.cpp, box_hit) does, but for an origin whose
only NaN is in y, for which that reports a NaN distance. A hit within the range must be found however
close to it the range ends: the boxes' entry distances and the hit distance are rounded separately, so
the traversal may discard a box only with a margin.
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


def quad(axis, at, side):
    """A square of two right-angled triangles in the plane x[axis] = at, about the axis."""
    u, v = (axis + 1) % 3, (axis + 2) % 3
    prims = np.zeros(2, pa.PRIM_DTYPE)
    for p, s in zip(prims, (side, -side)):
        for name, (a, b) in (("p0", (-s, -s)), ("p1", (s, -s)), ("p2", (-s, s))):
            p[name][u], p[name][v], p[name][axis] = a, b, at
    prims["light"] = prims["mediumInside"] = prims["mediumOutside"] = -1
    mats = np.zeros(1, pa.MATERIAL_DTYPE)
    mats["albedo"] = 0
    mats["albedoB"] = -1
    spec = np.zeros(1, pa.SPECTRUM_DTYPE)
    spec["scale"] = 1
    cam = pa.CameraEx()
    cam.width = cam.height = 8
    return pa.Scene(prims, mats, spec, None, None, camera=cam)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_range_one_float_above_the_hit(plugin, axis):
    # Against these triangles the hit distance takes six roundings that the box's entry distance does not
    # share (det 2, its reciprocal, the numerator 2, the product) and the entry distance two (the
    # reciprocal, the product): they are within 8 x 2^-24 = 4.8e-7 of each other, less than the traversal's
    # margin (1.5e-6). The rays stay inside the square: no other plane of the box is near the hit.
    rng = np.random.default_rng(axis)
    u, v = (axis + 1) % 3, (axis + 2) % 3
    n = 100000
    for at in (0.7, -3.3, 17.9):
        s = quad(axis, at, 121.7)
        rays = np.zeros(n, pa.RAY_DTYPE)
        rays["o"][:, u], rays["o"][:, v] = rng.uniform(-4, 4, (2, n))
        away = rng.choice([-1.0, 1.0], n)
        rays["o"][:, axis] = at + away * rng.uniform(0.1, 10, n)
        d = rng.normal(size=(n, 3))
        d[:, axis] = -away * (0.3 * np.linalg.norm(d, axis=1) + np.abs(d[:, axis]))  # at least 0.28 of the length below
        rays["d"] = d / np.linalg.norm(d, axis=1, keepdims=True)
        rays["tMax"] = np.inf
        far = plugin.trace(s, rays)
        on = far["prim"] >= 0  # a ray may pass between the two triangles
        assert on.mean() > 0.9999
        rays, far = rays[on], far[on]
        rays["tMax"] = np.nextafter(far["t"], np.float32(np.inf))
        assert np.array_equal(words(plugin.trace(s, rays)), words(far))
        assert np.all(plugin.trace(s, rays, any_hit=True)["prim"] >= 0)
        rays["tMax"] = far["t"]  # the range is open
        assert np.all(plugin.trace(s, rays)["prim"] < 0)
