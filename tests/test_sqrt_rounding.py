"""The rounding step of the device's square root of 1 - a (sqrt_1m, pt_common.h), restated in NumPy.

The hardware instruction is within one ulp of the root; two fused residuals then choose among it and
its neighbours. For every argument that 1 - a can take (zero, and 2^-24 up to 1) and each of the
three starts, the choice must be the correctly rounded root. The residuals' signs are exact in
double precision: a product of two float32 values fits it.
"""
import numpy as np
import pytest


def ulps(x, k):
    return (x.view(np.int32) + np.int32(k)).view(np.float32)


def rounded(x, s):
    lo, hi = ulps(s, -1), ulps(s, 1)
    res = lambda t: x.astype(np.float64) - t.astype(np.float64) * s.astype(np.float64)  # noqa: E731
    with np.errstate(invalid="ignore"):
        r = np.where(res(lo) <= 0, lo, s)
        return np.where(res(hi) > 0, hi, r)


@pytest.mark.parametrize("start", [-1, 0, 1])
def test_neighbours_round_to_the_root(start):
    k = np.arange(1, 1 << 24, 7, dtype=np.uint32)
    x = np.concatenate([(k * np.float64(2.0 ** -24)).astype(np.float32), np.float32(2.0) ** -np.arange(0, 25, dtype=np.float32)])
    root = np.sqrt(x.astype(np.float64)).astype(np.float32)
    assert np.array_equal(rounded(x, ulps(root, start)), root)


def test_zero_stays_zero():
    x = np.zeros(1, np.float32)
    assert rounded(x, x)[0] == 0
