"""The kernels' Snake (snake.h), compiled for the host, against 64 bits: the reduction, the polynomial and the
branch for large arguments, over every range they are used on.

Bound of one value: the result is at most 1, so its own rounding is half a unit of 2^-24, and what rounding
r, z and z^2 leaves is at most as much each (|r| <= pi / 4): 1.2e-7 in all. Over many values the error
has to be no larger than that of a correctly rounded sinf, squared in f32, which it stands for.
"""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

F = np.float32
NATIVE = Path(__file__).resolve().parent / "native"
BOUND = 1.2e-7


@pytest.fixture(scope="module")
def lib():
    so = NATIVE / "lib" / "libsnake.so"
    if not so.exists():
        subprocess.run(["make", "-s", "-C", str(NATIVE), str(so)], check=True)
    L = ctypes.CDLL(str(so))
    L.sin2_max.restype = ctypes.c_float
    return L


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _sin2(lib, u, wide=False):
    u, out = np.ascontiguousarray(u, F), np.empty(len(u), F)
    lib.sin2_values(_ptr(u), len(u), int(wide), _ptr(out))
    return out


def _snake16(lib, v, za, zb):
    v, out = np.ascontiguousarray(v, F), np.empty(16, F)
    lib.snake16(_ptr(v), ctypes.c_float(za), ctypes.c_float(zb), _ptr(out))
    return out


def _rms(x):
    return float(np.sqrt(np.mean(np.square(x))))


@pytest.mark.parametrize("scale", [1e-3, 0.1, 0.3, 1.0, 3.0, 30.0, 1e4, 2.5e5])
def test_sin2_is_as_exact_as_sinf_squared(lib, scale):
    u = (np.random.default_rng(1).standard_normal(200000) * scale).astype(F)
    u = u[np.abs(u) <= lib.sin2_max()]
    want = np.sin(u.astype(np.float64)) ** 2
    rounded = np.sin(u.astype(np.float64)).astype(F)
    err = _sin2(lib, u) - want
    assert np.abs(err).max() < BOUND
    assert _rms(err) <= _rms(rounded * rounded - want)
    small = np.abs(u) < 1e-2
    assert np.allclose(_sin2(lib, u)[small], want[small], rtol=5e-7, atol=0)


# 64-bit sin holds its phase over all of these; past 2.8e16 one pass alone would leave the polynomial's range
@pytest.mark.parametrize("scale", [2.0 ** 20, 1e9, 1e13, 2e16, 1e17, 1e20, 1e23])
def test_sin2_wide_reduction(lib, scale):
    u = (np.random.default_rng(2).uniform(1, 4, 3000) * scale).astype(F)
    want = np.sin(u.astype(np.float64)) ** 2
    rounded = np.sin(u.astype(np.float64)).astype(F)
    err = _sin2(lib, u, wide=True) - want
    assert np.abs(err).max() < BOUND
    assert _rms(err) <= _rms(rounded * rounded - want)


def test_sin2_past_the_phases_reach(lib):
    """Past 2^80 the value is some sin^2 all the same; infinities and NaN have none."""
    got = _sin2(lib, np.array([1e30, -3.4028234e38, 3.4028234e38], F), wide=True)
    assert ((got >= 0) & (got <= 1 + BOUND)).all()
    assert np.isnan(_sin2(lib, np.array([np.inf, -np.inf, np.nan], F), wide=True)).all()
    assert np.isnan(_sin2(lib, np.array([np.nan], F))).all()


@pytest.mark.parametrize("za,zb", [(1.0, 1.0), (0.37, 2.5), (3.0e4, 0.01)])
def test_snake_of_mixed_arguments(lib, za, zb):
    """Small and large arguments of either sign, both sides of the limit, and NaN among the values of one
    lane: each is what it is alone."""
    lim = lib.sin2_max()
    edge = [np.nextafter(F(lim), F(0)), F(lim), np.nextafter(F(lim), F(np.inf)), F(4 * lim)]
    vals = np.array([0.0, 1e-3, -0.5, 1.5, -7.0, 300.0, *edge, *[-x for x in edge], 1e12, np.nan], F)
    v = (vals / F(za)).astype(F)
    got = _snake16(lib, v, za, zb)
    u = (v * F(za)).astype(F)
    want = v.astype(np.float64) + np.sin(u.astype(np.float64)) ** 2 * np.float64(F(zb))
    ok = np.isfinite(v)
    bound = zb * BOUND + np.abs(want[ok]) * 2.0 ** -24
    assert (np.abs(got[ok] - want[ok]) <= bound).all()
    assert np.isnan(got[~ok]).all()
    # without the large ones the lane takes the other branch: the same values
    few = np.where(np.abs(u) <= lim, v, F(0))
    small = np.abs(u) <= lim
    np.testing.assert_array_equal(_snake16(lib, few, za, zb)[small], got[small])
    inf = v.copy()
    inf[3] = np.inf
    assert np.isnan(_snake16(lib, inf, za, zb)[3])
