"""The kernels' two-instruction quotient (bf_device.hip.h: quot_by / quot): fma(v, hi, v * lo) against the
correctly rounded v / sa, at every pair of operands where the two could fall on different sides of a
quantiser's decision.

A quantiser rounds fl(v / sa) to an integer (or to an e4m3 value), so only the side of a midpoint h matters,
and fl(v / sa) changes sides at h +- half a unit in the last place of h.  hi + lo is 1 / sa to about
2^-48, so an operand pair can only go wrong if its quotient lies within a few 2^-48 of such an edge M:
with significands V, S (24 bits) and m (25 bits, odd) that is |V * 2^a - m * S| <= 16, and for each m and
each difference there is at most one S modulo 2^a.  They are enumerated here in exact arithmetic.
"""
from fractions import Fraction as F

import numpy as np


def _round32(x: F) -> F:
    """Nearest fp32 (normal range), ties to even, of an exact rational."""
    if x == 0:
        return F(0)
    sign, x = (-1, -x) if x < 0 else (1, x)
    e = x.numerator.bit_length() - x.denominator.bit_length()
    if F(2) ** e > x:
        e -= 1
    u = F(2) ** (e - 23)
    n, r = divmod(x, u)
    n = int(n)
    if 2 * r > u or (2 * r == u and n & 1):
        n += 1
    return sign * n * u


def _quot(v: F, sa: F) -> F:
    """quot(v, quot_by(sa)) as the device computes it; the reciprocal is correctly rounded (recip, which
    tests/test_quotient_gpu.py holds to that on the device)."""
    hi = _round32(1 / sa)
    rem = _round32(1 - sa * hi)
    lo = _round32(rem * hi + _round32(_round32(rem * hi) * (rem / 2)))
    return _round32(v * hi + _round32(v * lo))


def _midpoints():
    ints = {F(2 * k + 1, 2) for k in range(256)}
    e4m3 = sorted({F(m, 8) * F(2) ** -6 for m in range(8)} | {(1 + F(m, 8)) * F(2) ** e for m in range(8) for e in range(-6, 9)})
    return ints | {(a + b) / 2 for a, b in zip(e4m3, e4m3[1:])}


def _edges(h: F):
    """The odd 25-bit significand m and exponent of the two edges of h's rounding interval."""
    e = h.numerator.bit_length() - h.denominator.bit_length()
    if F(2) ** e > h:
        e -= 1
    half = F(2) ** (e - 24)
    for edge in (h + half, h - (half / 2 if h == F(2) ** e else half)):
        m, j = edge, 0
        while m.denominator > 1:
            m, j = m * 2, j - 1
        m = int(m)
        while m % 2 == 0:
            m, j = m // 2, j + 1
        yield m, j


def test_the_quotient_falls_on_the_same_side_of_every_midpoint():
    pairs = set()
    for h in _midpoints():
        for m, j in _edges(h):
            for a in (23, 24, 25, 26):
                mod = 1 << a
                inv = pow(m, -1, mod)
                for d in range(-16, 17):
                    s = (-d * inv) % mod if d else 0
                    while 0 < s < 1 << 24:
                        big = m * s + d
                        if s >= 1 << 23 and big % mod == 0 and 1 << 23 <= big >> a < 1 << 24:
                            v, sa = F(big >> a) * F(2) ** (a + j), F(s)
                            want, got = _round32(v / sa), _quot(v, sa)
                            assert (want < h, want > h) == (got < h, got > h), (float(h), s, big >> a, d)
                            pairs.add((s, big >> a))
                        s += mod
    assert len(pairs) > 1000


def test_the_quotient_near_random_ties():
    rng = np.random.default_rng(0)
    for _ in range(4000):
        sa, k = F(int(rng.integers(1 << 23, 1 << 24))), int(rng.integers(0, 255))
        h = F(2 * k + 1, 2)
        v = _round32(sa * h)                       # the operand nearest to the tie (the tie itself for short scales)
        want, got = _round32(v / sa), _quot(v, sa)
        assert (want < h, want > h) == (got < h, got > h), (v, sa)
