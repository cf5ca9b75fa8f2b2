"""The persistent traversal's ray feed and stack at the sizes where they change behaviour.

A ray's hit does not depend on the batch it is traced in, so a large batch (runs of one size per
wave, dealt tiles, tiles from the device counters, a ragged last tile) must equal, bit for bit, the
same rays traced in small ones, which take the other branch and are checked against the oracle in
test_trace_gpu.py. A stack of parallel sheets makes every node's eight children pending at once:
traversal stacks that spill to device memory. The expected hits are the sheets' own order.
"""
import numpy as np
import pytest

import prender_amd as pa
import raygen

pytestmark = pytest.mark.gpu

LANES = 256 * 8 * 256  # lanes of the largest traversal launch on a 256-CU device


@pytest.fixture(scope="module")
def rays(c1):
    lo, hi = raygen.scene_bounds(c1)
    r = raygen.random_rays(lo, hi, 4 * LANES + 4 * 64 + 37, 11)
    r["tMax"][::5] = 3.0
    return r


@pytest.fixture(scope="module")
def small_batches(plugin, c1, rays):
    parts = [(plugin.trace(c1, rays[i:i + 40000]), plugin.trace(c1, rays[i:i + 40000], any_hit=True)["prim"] >= 0)
             for i in range(0, len(rays), 40000)]
    return np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 2047, 2048, 2049, 131071, 131073, LANES - 1, LANES, LANES + 1,
                               2 * LANES - 63, 2 * LANES + 65, 4 * LANES + 4 * 64 + 37])
def test_batch_sizes(plugin, c1, rays, small_batches, n):
    got = plugin.trace(c1, rays[:n])
    assert got.tobytes() == small_batches[0][:n].tobytes()
    assert np.array_equal(plugin.trace(c1, rays[:n], any_hit=True)["prim"] >= 0, small_batches[1][:n])


def sheets(n):
    """n sheets (two triangles each) in the planes z = 1 .. n, in shuffled order."""
    order = np.random.default_rng(3).permutation(n)
    prims = np.zeros(2 * n, pa.PRIM_DTYPE)
    for half, (a, b) in enumerate((((9, -9), (9, 9)), ((9, 9), (-9, 9)))):
        p = prims[half::2]
        z = (1.0 + order).astype(np.float32)
        for name, (x, y) in (("p0", (-9, -9)), ("p1", a), ("p2", b)):
            p[name][:, 0], p[name][:, 1], p[name][:, 2] = x, y, z
    prims["light"] = prims["mediumInside"] = prims["mediumOutside"] = -1
    mats = np.zeros(1, pa.MATERIAL_DTYPE)
    mats["albedo"] = 0
    mats["albedoB"] = -1
    spec = np.zeros(1, pa.SPECTRUM_DTYPE)
    spec["scale"] = 1
    cam = pa.CameraEx()
    cam.width = cam.height = 8
    return pa.Scene(prims, mats, spec, None, None, camera=cam), order


@pytest.mark.parametrize("n", [5, 64, 3000])
def test_deep_stacks(plugin, n):
    s, order = sheets(n)
    rng = np.random.default_rng(n)
    m = 4099
    rays = np.zeros(m, pa.RAY_DTYPE)
    rays["o"][:, :2] = rng.uniform(-4, 4, (m, 2))
    start = rng.integers(0, n + 1, m)  # between the sheets start and start + 1 (z = start + 0.5)
    rays["o"][:, 2] = start + 0.5
    up = rng.random(m) < 0.5
    rays["d"][:, 2] = np.where(up, 1, -1)
    rays["tMax"] = np.inf
    plane = np.where(up, start + 1, start)
    hit = (plane >= 1) & (plane <= n)
    got = plugin.trace(s, rays)
    assert np.array_equal(got["prim"] >= 0, hit)
    assert np.array_equal(got["t"], np.where(hit, np.float32(0.5), np.float32(0)))
    assert np.array_equal(order[got["prim"][hit] // 2] + 1, plane[hit])
    # any hit: a range that ends before the nearest sheet, or reaches it
    rays["tMax"] = np.where(rng.random(m) < 0.5, 0.25, 0.75)
    occ = plugin.trace(s, rays, any_hit=True)["prim"] >= 0
    assert np.array_equal(occ, hit & (rays["tMax"] > 0.5))
