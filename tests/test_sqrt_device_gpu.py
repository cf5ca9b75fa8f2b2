"""sqrt_1m (pt_common.h) on the device: the root of 1 - a must be the correctly rounded one, bit for
bit, for every value that 1 - a takes for a in [0, 1] (the multiples of 2^-24), and for a below zero, above
one, infinite and NaN what the library square root gives (test_sqrt_rounding.py shows why the rounding
step suffices). tests/device_probe is built with the other native code.
"""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def probe(plugin):
    lib = C.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "device_probe", "libprobe.so"))

    def run(a):
        a = np.ascontiguousarray(a, np.float32)
        out, plain = np.zeros_like(a), np.zeros_like(a)
        p = lambda x: x.ctypes.data_as(C.c_void_p)  # noqa: E731
        assert lib.probe_sqrt_1m(p(a), p(out), p(plain), len(a)) == 0
        return out, plain

    return run


def root(x):  # float64's root, rounded to float32, is the correctly rounded one
    return np.sqrt(x.astype(np.float64)).astype(np.float32)


def test_every_difference_from_one(probe):
    x = (np.arange((1 << 24) + 1) * 2.0 ** -24).astype(np.float32)
    a = np.float32(1) - x
    assert np.array_equal(np.float32(1) - a, x)
    out, plain = probe(a)
    assert np.array_equal(out.view(np.int32), root(x).view(np.int32))
    assert np.array_equal(plain.view(np.int32), out.view(np.int32))


def test_outside_of_the_unit_interval(probe):
    rng = np.random.default_rng(1)
    a = np.concatenate([-np.exp2(rng.uniform(-26, 127.9, 1 << 20)), np.exp2(rng.uniform(0, 127.9, 1000)),
                        [0.0, -0.0, 1.0, np.nextafter(np.float32(1), np.float32(2)), 1e-30, -1e-30, np.inf, -np.inf,
                         np.nan, 3.4028235e38, -3.4028235e38]]).astype(np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        x = np.float32(1) - a
    out, plain = probe(a)
    assert np.array_equal(out.view(np.int32), root(np.where(x > 0, x, np.float32(0))).view(np.int32))
    assert np.array_equal(plain.view(np.int32), out.view(np.int32))
