"""hypot_key of csrc/bla_key.hpp, restated: within [2^-480, 2^500] the bits of
x^2 + y^2 are the key that the prescaled squares give, down to a smaller
component whose square is subnormal or zero."""
import math
import struct

import numpy as np
import pytest


def bits(x):
    return struct.unpack("<q", struct.pack("<d", x))[0]


def prescaled(x, y):
    e = math.frexp(max(abs(x), abs(y)))[1] - 1
    xs, ys = math.ldexp(x, -e), math.ldexp(y, -e)
    return bits(xs * xs + ys * ys) + e * (1 << 53)


@pytest.mark.parametrize("scale", [-480, -479, -470, -450, -300, 0, 300, 498, 499])
def test_direct_key(scale):
    rng = np.random.default_rng(scale + 1000)
    for _ in range(300):
        x = math.ldexp(1. + rng.random(), scale)
        for down in (0, 1, 5, 25, 26, 27, 28, 31, 40, 51, 53, 54, 60, 64, 300):
            y = math.ldexp(rng.random() - 0.5, scale - down)
            for u, v in ((x, y), (y, x), (-x, y)):
                assert bits(u * u + v * v) == prescaled(u, v)
    for x in (math.ldexp(1., -480), math.ldexp(2. - 2.**-52, -480), math.ldexp(1., 500)):
        assert bits(x * x) == prescaled(x, 0.)
