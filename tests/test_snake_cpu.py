"""The Snake's sin^2 (conv.h sin2_*) restated in numpy f32 against 64 bits: the pi reduction and the
polynomial over every range they are used on. Bound: the result is at most 1, so its own rounding and
that of its last product allow about two units of 2^-24 each way, 2.5e-7; the reduction adds the rounding
of r (half a unit of 1.6, times a slope of at most 1).
"""
import re
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

F = np.float32
SRC = (Path(__file__).resolve().parent.parent / "navi-tts_amd" / "csrc" / "hip" / "conv.h").read_text()


def _fma(a, b, c):
    return (np.asarray(a, np.float64) * np.asarray(b, np.float64) + np.asarray(c, np.float64)).astype(F)


def _coefficients():
    body = SRC[SRC.index("float sin2_poly(float r)"):]
    body = body[:body.index("}")]
    return [F(x) for x in re.findall(r"(-?\d\.\d+(?:e-?\d+)?)f", body)]


def _poly(r):
    z = (r * r).astype(F)
    c = _coefficients()
    p = np.full_like(z, c[0])
    for k in c[1:]:
        p = _fma(p, z, k)
    return _fma((z * z).astype(F), p, z)


@pytest.mark.parametrize("scale", [1e-3, 0.1, 1.0, 30.0, 1e4, 2.5e5])
def test_sin2_f32_reduction(scale):
    u = (np.random.default_rng(1).standard_normal(200000) * scale).astype(F)
    u = u[np.abs(u) <= 2 ** 20]
    n = np.rint((u * F(0.318309873)).astype(F)).astype(F)
    got = _poly(_fma(-n, F(-8.74227766e-8), _fma(-n, F(3.14159274), u)))
    want = np.sin(u.astype(np.float64)) ** 2
    assert len(_coefficients()) == 6
    assert np.abs(got - want).max() < 3e-7
    small = np.abs(u) < 1e-2
    assert np.allclose(got[small], want[small], rtol=5e-7, atol=0)


def _wide(u):
    """One argument of sin2_reduce_wide: three passes, their fma sums exact before they are rounded."""
    r = float(u)
    for _ in range(3):
        m = Fraction(float(np.rint(np.float64(r) * 0.3183098861837907)))
        t = float(Fraction(r) - m * Fraction(3.141592653589793))
        r = float(Fraction(t) - m * Fraction(1.2246467991473532e-16))
    return F(r)


# 64-bit sin holds its phase over all of these; past 2.8e16 one pass alone would leave the polynomial's range
@pytest.mark.parametrize("scale", [2.0 ** 20, 1e9, 1e13, 2e16, 1e17, 1e20, 1e23])
def test_sin2_wide_reduction(scale):
    u = (np.random.default_rng(2).uniform(1, 4, 300) * scale).astype(F)
    r = np.array([_wide(x) for x in u])
    assert np.abs(r).max() < 1.64
    want = np.sin(u.astype(np.float64)) ** 2
    assert np.abs(_poly(r) - want).max() < 3e-7


@pytest.mark.parametrize("u", [1e30, -3.4028234e38])
def test_sin2_wide_reduction_is_bounded(u):
    """Past the phase's reach the value is some sin^2 all the same."""
    r = _wide(F(u))
    assert abs(r) < 1.64 and 0 <= _poly(np.array([r]))[0] <= 1 + 3e-7
