"""The shorter forms of ocfd_common.h that the FP64 path's bit identity rests
on, against the forms they stand for: the minmod limiters as medians, the
division by a divisor known in advance, the quotient of the WENO weights
without operand scaling, and the fused sums with power-of-two factors."""
import ctypes
import ctypes.util

import numpy as np
import pytest

_m = ctypes.CDLL(ctypes.util.find_library("m"))
_m.fma.restype = ctypes.c_double
_m.fma.argtypes = [ctypes.c_double] * 3
_m.fmaf.restype = ctypes.c_float
_m.fmaf.argtypes = [ctypes.c_float] * 3
fma, fmaf = _m.fma, lambda a, b, c: np.float32(_m.fmaf(a, b, c))


def values(rng, n):
    """Values of many magnitudes and both signs, zeros and equal neighbours."""
    x = rng.standard_normal(n) * 10.0 ** rng.uniform(-12, 12, n)
    x[rng.random(n) < 0.05] = 0.0
    same = rng.random(n) < 0.1
    x[1:][same[1:]] = x[:-1][same[1:]]
    return x


def minmod2(a, b):
    return 0.5 * (np.copysign(1.0, a) + np.copysign(1.0, b)) * np.minimum(abs(a), abs(b))


def minmod4(a, b, c, d):
    s = [np.copysign(1.0, v) for v in (a, b, c, d)]
    r = 0.5 * (s[0] + s[1]) * abs(0.5 * (s[0] + s[2])) * abs(0.5 * (s[0] + s[3]))
    return r * np.minimum.reduce([abs(v) for v in (a, b, c, d)])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_minmod_as_median(dtype):
    rng = np.random.default_rng(1)
    a, b, c, d = (values(rng, 200000).astype(dtype) for _ in range(4))
    assert np.array_equal(np.fmax(np.fmin(a, b), np.fmin(np.fmax(a, b), 0)), minmod2(a, b))
    lo, hi = np.fmin.reduce([a, b, c, d]), np.fmax.reduce([a, b, c, d])
    assert np.array_equal(np.fmax(lo, np.fmin(hi, 0)), minmod4(a, b, c, d))


@pytest.mark.parametrize("divisor", [3.0, 0.1, 0.5, 2.25, 2.8, 6.0, None])
def test_division_by_a_known_divisor(divisor):
    rng = np.random.default_rng(2)
    for a in values(rng, 20000):
        b = float(rng.uniform(1e-3, 1e3)) if divisor is None else divisor
        y = 1.0 / b
        q = a * y
        assert fma(fma(-b, q, a), y, q) == a / b
        a32, b32 = np.float32(a), np.float32(b)
        y32 = np.float32(1.0) / b32
        q32 = a32 * y32
        assert fmaf(fmaf(-b32, q32, a32), y32, q32) == a32 / b32


def test_weight_quotient_without_scaling():
    rng = np.random.default_rng(3)
    for s in 10.0 ** rng.uniform(-20, 30, 20000):
        b = (1.0e-8 + s) * (1.0e-8 + s)
        for a in (0.3, 18.0 / 35.0, float(rng.standard_normal())):
            y = (1.0 / b) * (1.0 + rng.uniform(-1, 1) * 2.0 ** -24)  # a reciprocal estimate
            for _ in range(2):
                y = fma(y, fma(-b, y, 1.0), y)
            q = a * y
            assert fma(fma(-b, q, a), y, q) == a / b


def test_fused_sums_with_power_of_two_factors():
    rng = np.random.default_rng(4)
    x, z = values(rng, 20000), values(rng, 20000)
    for k in (2.0, 4.0, 0.25, -0.5, -2.0):
        assert all(fma(k, p, q) == k * p + q for p, q in zip(x, z))
