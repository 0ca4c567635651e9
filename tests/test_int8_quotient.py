"""The 8-bit quantizer's quotient: x y, corrected once by its remainder, in place of the float32 division, where what follows
is a rounding to binary16."""
from fractions import Fraction

import numpy as np

F32, F16 = np.float32, np.float16


def _round24(v):
    """A positive rational to 24 significant bits, ties to even."""
    e = 0
    while v >= 1 << 24:
        v, e = v / 2, e + 1
    while v < 1 << 23:
        v, e = v * 2, e - 1
    n = int(v)
    rest = v - n
    n += rest > Fraction(1, 2) or (rest == Fraction(1, 2) and n & 1)
    return Fraction(n) * Fraction(2) ** e


def _signed_round24(v):
    return Fraction(0) if v == 0 else _round24(v) if v > 0 else -_round24(-v)


def test_no_quotient_beside_a_binary16_midpoint_is_missed():
    """The corrected product misses the correctly rounded quotient by its own error, below 2^-21 units in the last place, so only
    where X / S lies that close to a midpoint of float32; and after rounding to binary16 it shows only if that midpoint
    neighbours one of binary16.  With M that midpoint in half units (25 bits, odd), X 2^j = M S + d: all solutions with
    |d| <= 12, twice what the error allows."""
    seen = 0
    for m in range(1024):
        for side in (-1, 1):
            mid = (2 * (1024 + m) + 1 << 13) + side
            for j in (24, 25):
                inv = pow(mid, -1, 1 << j)
                for d in range(-12, 13):
                    S = -d * inv % (1 << j)
                    if d == 0 or not 1 << 23 <= S < 1 << 24:
                        continue
                    X = mid * S + d >> j
                    if not 1 << 23 <= X < 1 << 24:
                        continue
                    seen += 1
                    y = _round24(Fraction(1, S))
                    q0 = _round24(X * y)
                    q = _signed_round24(q0 + _signed_round24(X - q0 * S) * y)
                    want = _round24(Fraction(X, S))
                    if q != want:   # (half a unit apart at most: the same binary16 number is all that is needed)
                        scale = 2.0 ** 6
                        assert F16(float(q) * scale) == F16(float(want) * scale), (X, S)
    assert seen > 15000


def test_quotients_at_random():
    """The same statement on ordinary numbers, with the fused multiply-add formed in float64: exact but for the last sum, whose
    rounding there is far finer than what binary16 sees."""
    rng = np.random.default_rng(5)
    s = (rng.uniform(1, 2, 400000) * 2.0 ** rng.integers(-12, 4, 400000)).astype(F32)
    x = (s * rng.uniform(-130, 130, 400000)).astype(F32)
    y = (F32(1) / s).astype(F32)
    q0 = (x * y).astype(F32)
    r = (x.astype(np.float64) - q0.astype(np.float64) * s.astype(np.float64)).astype(F32)
    q = (q0.astype(np.float64) + r.astype(np.float64) * y.astype(np.float64)).astype(F32)
    assert np.array_equal(q.astype(F16), (x / s).astype(F16))
