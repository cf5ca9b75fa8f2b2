"""Device staging that outlives a call, and the content keys that decide what is resident.

Host films, sample records and the guiding probes' arrays go through buffers kept from call to call:
calls of changing size, with and without the sum of squares, must give what a first call gives. A
small scene, which the keys hash whole, changed in place, at the same addresses, must not be taken for the
resident one (larger ones: test_residency_gpu.py).
"""
import numpy as np
import pytest

import prender_amd as pa

pytestmark = pytest.mark.gpu

SIZES = [(64, 40), (17, 9), (33, 70), (1, 1), (64, 40)]


def params(first=0):
    return pa.render_params(spp=2, first_sample=first, seed=3, max_depth=4)


def test_host_films_of_changing_size(plugin, host):
    scenes = [host.generate(1, w, h, 0.25) for w, h in SIZES]
    fresh = []
    for s in scenes:
        plugin.release()
        fresh.append((plugin.render_ex(s, params()), plugin.sample_radiance(s, params()).tobytes()))
    for k in (0, 1, 2, 3, 4, 1, 0):
        s = scenes[k]
        film, sq = plugin.render_ex(s, params())
        only, none = plugin.render_ex(s, params(), variance=False)
        assert none is None
        assert np.array_equal(film, fresh[k][0][0]) and np.array_equal(sq, fresh[k][0][1]) and np.array_equal(only, film)
        assert plugin.sample_radiance(s, params()).tobytes() == fresh[k][1]


def test_guide_probes_of_changing_size(plugin):
    rng = np.random.default_rng(2)
    R = rng.random((1000, 16)).astype(np.float32)
    whole = plugin.guide_eval(R[:, :9])
    for n in (1, 1000, 37):
        assert np.array_equal(plugin.guide_eval(R[:n, :9]), whole[:n])
    g = plugin.guide_grad(R)[0]
    plugin.guide_grad(R[:5])
    assert np.allclose(plugin.guide_grad(R)[0], g, rtol=1e-4, atol=1e-6 * np.abs(g).max())


def test_scene_changed_in_place(plugin, host):
    s = host.generate(1, 32, 18, 0.25)
    before, _ = plugin.render_ex(s, params())
    scale = s.spectra["scale"].copy()
    s.spectra["scale"][s.lights["spectrum"]] *= 2  # the emitters' radiance
    twice, _ = plugin.render_ex(s, params())
    assert np.allclose(twice, 2 * before, rtol=1e-5, atol=1e-12) and before.any()
    s.spectra["scale"][:] = scale
    assert np.array_equal(plugin.render_ex(s, params())[0], before)
    s.prims["p0"][-1, 1] += 0.25  # one vertex: the geometry and everything after it
    moved, _ = plugin.render_ex(s, params())
    fresh = pa.Scene(s.prims.copy(), s.materials, s.spectra, s.knots, s.lights, s.media, s.grid, s.camera,
                     s.desc.cameraMedium, s.defaults)
    assert np.array_equal(moved, plugin.render_ex(fresh, params())[0])
