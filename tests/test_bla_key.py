"""The integer keys of csrc/bla_key.hpp, restated: modulus_key(q, e) <
radius_key(r) decides as sqrt(q) 2^e < r does, the comparison of the
reference's BLA lookup (perturbation.py:2116-2170), on both sides of every
radius, for subnormal, zero and infinite radii and for a zero z."""
import math
import struct

import numpy as np
import pytest

KEY_MIN_E, KEY_MAX_E = -1100, 511
INT64_MIN, INT64_MAX = -(1 << 63), (1 << 63) - 1


def bits(x):
    return struct.unpack("<q", struct.pack("<d", x))[0]


def of_bits(b):
    return struct.unpack("<d", struct.pack("<q", b))[0]


def radius_key(r):
    if not r > 0.:
        return INT64_MIN
    if math.isinf(r):
        return INT64_MAX
    m, e = math.frexp(r)
    m, e = 2. * m, e - 1
    if e >= KEY_MAX_E:
        return (1023 + 2 * KEY_MAX_E) << 52
    t = m * m
    while math.sqrt(t) >= m:
        t = of_bits(bits(t) - 1)
    while math.sqrt(t) < m:
        t = of_bits(bits(t) + 1)
    return bits(t) + e * (1 << 53)


def modulus_key(q, e):
    b = bits(q)
    hi = max(b >> 32, 0x3ff00000) + (min(max(e, KEY_MIN_E), KEY_MAX_E) << 21)
    key = (hi << 32) | (b & 0xffffffff)
    assert INT64_MIN <= key <= INT64_MAX
    return key


def below(q, e, r):
    """sqrt(q) 2^e < r, exactly; from 2^511 on (|z|^2 beyond binary64) below
    no finite radius."""
    if math.isinf(r):
        return True
    s = math.sqrt(q)
    if s == 0. or not r > 0.:
        return s == 0. and r > 0.
    if e >= KEY_MAX_E:
        return False
    m, er = math.frexp(r)
    ms, es = math.frexp(s)
    return (es + e, ms) < (er, m)


@pytest.mark.parametrize("scale", [0, -3, -500, -1000, -1022, -1050, -1073, 300, 505, 1000])
def test_key_decides_as_the_square_root(scale):
    rng = np.random.default_rng(scale + 5000)
    for _ in range(400):
        r = math.ldexp(1. + rng.random(), scale)
        m, e = math.frexp(r)
        m, e = 2. * m, e - 1
        rk = radius_key(r)
        for d in range(-4, 5):                       # q around the square of the radius's mantissa
            q = of_bits(bits(m * m) + d)
            if q >= 1.:
                assert (modulus_key(q, e) < rk) == below(q, e, r)
                assert (modulus_key(2. * q, e) < rk) == below(2. * q, e, r)
        for de in (-2000, -60, -1, 0, 1, 60):        # and far from it
            q = 1. + 7. * rng.random()
            assert (modulus_key(q, e + de) < rk) == below(q, e + de, r)


@pytest.mark.parametrize("r", [1., 2., 0.5, 5e-324, 1e-320, 2.2250738585072014e-308, 1.7976931348623157e308])
def test_key_at_powers_of_two_and_range_ends(r):
    m, e = math.frexp(r)
    m, e = 2. * m, e - 1
    for d in range(-3, 4):
        q = of_bits(bits(m * m) + d)
        if q >= 1.:
            assert (modulus_key(q, e) < radius_key(r)) == below(q, e, r)
    assert modulus_key(0., -(1 << 26)) < radius_key(r)      # z = 0 carries the zero exponent


def test_key_of_zero_and_infinite_radius():
    for q, e in ((0., -(1 << 26)), (1., -7000), (1., -1100), (3., 0), (7., 1000)):
        assert not modulus_key(q, e) < radius_key(0.)
        assert not modulus_key(q, e) < radius_key(float("nan"))
        assert modulus_key(q, e) < radius_key(float("inf"))
    assert not modulus_key(float("nan"), 0) < radius_key(1e300)
