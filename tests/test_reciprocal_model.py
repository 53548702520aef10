"""Error model of the FP64 root, reciprocal root and reciprocal of the force
passes (sqrt_rsqrt and fast_rcp), step by step in exact arithmetic rounded
once per operation, from estimates as far off as the hardware's (2^-24) and
twice that: the root of a squared distance and the reciprocals come out
rounded to nearest, as the library's root and division, over the distances and
the r/sigma - a that the passes meet."""
from fractions import Fraction
import math
import random

EST = 2.0 ** -23


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))  # (int / int rounds to nearest)


def _estimate(v, rng):
    """v off by at most EST, in 26 bits."""
    y = v * (1.0 + rng.uniform(-EST, EST))
    m, e = math.frexp(y)
    return math.ldexp(round(m * 2 ** 26), e - 26)


def sqrt_rsqrt(a, y):
    g, h = a * y, 0.5 * y
    e = _fma(-h, g, 0.5)
    g, h = _fma(g, e, g), _fma(h, e, h)
    g = _fma(_fma(-g, g, a), h, g)
    s = _fma(_fma(-g, g, a), h, g)
    y1 = h + h
    return s, _fma(y1, _fma(-s, y1, 1.0), y1)


def fast_rcp(x, y):
    y = _fma(y, _fma(-x, y, 1.0), y)
    return _fma(y, _fma(-x, y, 1.0), y)


def _ulps(got, want):
    """Error of a double against an exact value, in units of its last place."""
    return abs(Fraction(got) - want) / Fraction(math.ulp(got))


def test_root_and_reciprocal_root():
    rng = random.Random(5)
    for k in range(4000):
        # metres, or units of sigma
        r = 10.0 ** rng.uniform(-12.0, -8.5) if k % 2 else rng.uniform(0.01, 3.0)
        a = r * r * (1.0 + rng.random())
        s, si = sqrt_rsqrt(a, _estimate(1.0 / math.sqrt(a), rng))
        assert s == math.sqrt(a)
        assert _ulps(si, 1 / Fraction(s)) <= Fraction(501, 1000)


def test_reciprocal():
    rng = random.Random(6)
    for k in range(4000):
        # r/sigma - a: -1.8 to -0.0018
        x = -1.8 * 10.0 ** rng.uniform(-3.0, 0.0) if k % 2 else rng.uniform(-1.85, -0.0017)
        y = fast_rcp(x, _estimate(1.0 / x, rng))
        assert _ulps(y, 1 / Fraction(x)) <= Fraction(501, 1000)
