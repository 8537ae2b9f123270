"""csrc/bla_key.hpp itself, compiled for the host: its keys are those of the
Python models that test_bla_key.py and test_bla_key_direct.py check, and decide
as the square root does."""
import math

import numpy as np
import pytest

import host_rules
import test_bla_key as model
from test_bla_key_direct import prescaled

def below(q, e, r):
    """The decision: the square root's, but from 2^511 on (|z|^2 beyond binary64)
    |z| is under no finite radius (bla_key.hpp)."""
    if math.isfinite(r) and math.log2(q) / 2 + e >= model.KEY_MAX_E:
        return False
    return model.below(q, e, r)


SCALES = [0, -3, -500, -1000, -1022, -1050, -1073, 300, 505, 511, 1000, 1023]


@pytest.mark.parametrize("scale", SCALES)
def test_radius_and_modulus_keys(scale):
    lib = host_rules.load()
    rng = np.random.default_rng(scale + 7000)
    for _ in range(200):
        r = math.ldexp(1. + rng.random(), scale)
        rk = lib.radius_key(r)
        assert rk == model.radius_key(r)
        m, e = math.frexp(r)
        m, e = 2. * m, e - 1
        for d in range(-4, 5):
            q = model.of_bits(model.bits(m * m) + d)
            if q >= 1.:
                assert lib.modulus_key(q, e) == model.modulus_key(q, e)
                assert (lib.modulus_key(q, e) < rk) == below(q, e, r)
        for de in (-2000, -60, -1, 0, 1, 60, 3000):
            q = 1. + 7. * rng.random()
            assert lib.modulus_key(q, e + de) == model.modulus_key(q, e + de)
            assert (lib.modulus_key(q, e + de) < rk) == below(q, e + de, r)


def test_range_ends():
    lib = host_rules.load()
    for r in (0., -1., float("nan"), float("inf"), 5e-324, 1e-320, 2.2250738585072014e-308, 1.7976931348623157e308,
              2.**511, math.nextafter(2.**511, 0.)):
        assert lib.radius_key(r) == model.radius_key(r)
    for q, e in ((0., -(1 << 26)), (1., -7000), (1., -1100), (3., 0), (7., 511), (7., 1000)):
        assert lib.modulus_key(q, e) == model.modulus_key(q, e)
    assert lib.modulus_key(0., -(1 << 26)) < lib.radius_key(5e-324)
    assert not lib.modulus_key(float("nan"), 0) < lib.radius_key(1e300)


@pytest.mark.parametrize("scale", [-1074, -1060, -1000, -901, -900, -899, -700, -481, -480, -479, -300, 0, 300, 499])
def test_hypot_key(scale):
    """The prescaled squares' key down to 2^-900; below it, and past 2^500, the
    key of the rounded modulus, which lies under the same radii."""
    lib = host_rules.load()
    rng = np.random.default_rng(scale + 9000)
    for _ in range(200):
        x = math.ldexp(1. + rng.random(), scale)
        for down in (0, 1, 26, 27, 53, 54, 64, 300):
            y = math.ldexp(rng.random() - 0.5, scale - down)
            for u, v in ((x, y), (y, x), (-x, y), (x, 0.)):
                if max(abs(u), abs(v)) >= 2.**-900:
                    assert lib.hypot_key(u, v) == prescaled(u, v)
                h = math.hypot(u, v)
                for r in (h * 0.999, h * 1.001, 2. * h, 0.5 * h):
                    if abs(r - h) > 1e-323:                # apart from ties of subnormal values
                        assert (lib.hypot_key(u, v) < lib.radius_key(r)) == (h < r)


def test_hypot_key_of_zero_huge_and_nan():
    lib = host_rules.load()
    inf, nan = float("inf"), float("nan")
    assert lib.hypot_key(0., 0.) < lib.radius_key(5e-324) and not lib.hypot_key(0., 0.) < lib.radius_key(0.)
    assert not lib.hypot_key(nan, nan) < lib.radius_key(inf) and not lib.hypot_key(inf, 1.) < lib.radius_key(inf)
    for x, y in ((nan, 1.), (1., nan), (nan, nan), (inf, 1.)):
        assert not lib.hypot_key(x, y) < lib.radius_key(1.7976931348623157e308)
    assert lib.hypot_key(1e300, 1.) < lib.radius_key(inf)
