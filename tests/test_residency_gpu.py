"""What a call takes for the scene already on the device (the content keys of api.hip and pt.hip).

Large arrays enter the key by their address and a sample of their elements: another buffer is another
scene even where it agrees at every sampled element, and after a change in place prgpu_release makes the
next call upload the scene again.
"""
import numpy as np
import pytest

import prender_amd as pa

pytestmark = pytest.mark.gpu

P = pa.render_params(spp=2, first_sample=0, seed=3, max_depth=16)


def with_grid(s, grid):
    return pa.Scene(s.prims, s.materials, s.spectra, s.knots, s.lights, s.media, grid, s.camera, s.desc.cameraMedium,
                    s.defaults)


def stride(count):  # every stride-th element of a large array is in the key
    return max(1, count // 4096)


def test_another_grid_that_agrees_at_the_samples(plugin, host):
    s = host.generate(3, 48, 27, 0.25)
    step = stride(len(s.grid))
    assert step > 1
    thin = np.zeros_like(s.grid)
    thin[::step] = s.grid[::step]
    dense = plugin.render_ex(s, P)[0]
    got = plugin.render_ex(with_grid(s, thin), P)[0]
    plugin.release()
    want = plugin.render_ex(with_grid(s, thin), P)[0]
    assert not np.array_equal(dense, want)
    assert np.array_equal(got, want)


def test_release_after_a_change_in_place(plugin, host):
    s = host.generate(1, 48, 27, 1.0)
    step = stride(len(s.prims))
    assert step > 1
    before = plugin.render_ex(s, P)[0]
    unsampled = np.arange(len(s.prims)) % step != 0
    unsampled[-1] = False
    for name in ("p0", "p1", "p2"):
        s.prims[name][unsampled, 1] += np.float32(0.25)
    plugin.release()
    after = plugin.render_ex(s, P)[0]
    fresh = pa.Scene(s.prims.copy(), s.materials, s.spectra, s.knots, s.lights, s.media, s.grid, s.camera,
                     s.desc.cameraMedium, s.defaults)
    assert not np.array_equal(after, before)
    assert np.array_equal(after, plugin.render_ex(fresh, P)[0])
