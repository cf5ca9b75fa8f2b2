"""The kernel variants of scenes that have media or interfaces but not both, against the oracle: the
sphere pyramid inside a fog that no interface bounds, and configuration 3 with every medium removed, whose
box is then an interface around nothing. (Scenes with both: test_media_gpu.py.)
"""
import numpy as np
import pytest

import prender_amd as pa
from test_pt_gpu import check_samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [0.0, 0.7])
def test_media_without_interfaces(plugin, host, g):
    s = host.generate(1, 64, 48, 0.25)
    spectra = np.concatenate([s.spectra, np.zeros(2, s.spectra.dtype)])
    spectra["kind"][-2:] = pa.SPEC_CONSTANT
    spectra["scale"][-2:] = 1
    spectra["p"][-2:, 0] = (0.02, 0.1)
    media = np.zeros(1, pa.MEDIUM_DTYPE)
    media["kind"] = pa.MEDIUM_HOMOGENEOUS
    media["sigmaA"], media["sigmaS"], media["scale"], media["g"] = len(s.spectra), len(s.spectra) + 1, 1, g
    prims = s.prims.copy()
    prims["mediumInside"] = prims["mediumOutside"] = 0
    fog = pa.Scene(prims, s.materials, spectra, s.knots, s.lights, media, None, s.camera, 0, s.defaults)
    for first in (0, 7):
        gpu, _ = check_samples(f"fog g={g}", fog, pa.render_params(spp=1, first_sample=first, seed=1, max_depth=32), plugin,
                               0.99)
        assert np.any(gpu["L"] > 0)


def test_interfaces_without_media(plugin, host):
    s = host.generate(3, 96, 54, 0.125)
    prims = s.prims.copy()
    prims["mediumInside"] = prims["mediumOutside"] = -1
    bare = pa.Scene(prims, s.materials, s.spectra, s.knots, s.lights, s.media, s.grid, s.camera, -1, s.defaults)
    for first in (0, 7):
        gpu, _ = check_samples("interfaces", bare, pa.render_params(spp=1, first_sample=first, seed=1, max_depth=32), plugin,
                               0.99)
        assert np.any(gpu["L"] > 0)
