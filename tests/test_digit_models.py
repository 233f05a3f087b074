"""CPU models of the digits that the split-precision kernels form, with exact rationals as reference.

* FP16 / BF16 digits by integer fields (PairDigits in split_f64.hip): one addition rounds a scaled
  value to an integer whose biased low word holds three digits.  The digits stay within the
  bounds that the level sums are proved with and reconstruct the value to half a unit of the last one.
* int8 digits by two FP64 additions (RowCut and digit_word in split_i8.hip): the balanced bytes of
  the value rounded to nearest, ties to even, in every row exponent's scaling.
"""
from fractions import Fraction

import numpy as np
import pytest

ROUND = 6755399441055744.0  # 1.5 x 2^52


def bits(x):
    return int(np.frombuffer(np.float64(x).tobytes(), np.uint64)[0])


def double(b):
    return float(np.frombuffer(np.uint64(b).tobytes(), np.float64)[0])


def low_word(x):
    return bits(x) & 0xFFFFFFFF


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))  # one rounding, to nearest even


def triple(u, beta):
    if beta == 9:
        return [((u >> 16) >> 2) - 512, ((u >> 9) & 511) - 256, (u & 511) - 256]
    return [(u - (1 << 32) if u >> 31 else u) >> 16, ((u >> 8) & 255) - 128, (u & 255) - 128]


def pair_digits(a, beta, S):
    """Digits of a = x 2^(3 BETA - e), step for step."""
    bias = (512 << 18) + (256 << 9) + 256 if beta == 9 else (128 << 8) + 128
    M, W = ROUND + bias, 2.0 ** (3 * beta)
    t = a + M
    d = triple(low_word(t), beta)
    r = a - (t - M)
    s = fma(r, W, M)
    d += triple(low_word(s), beta)
    if S == 7:
        q = fma(r, W, -(s - M))
        last = 512 if beta == 9 else 0
        f = low_word(fma(q, 2.0 ** beta, ROUND + last)) & 0xFFFF if beta == 9 else low_word(fma(q, 2.0 ** beta, ROUND))
        d.append(f - last if beta == 9 else (f - (1 << 32) if f >> 31 else f))
    return d


def values(rng, e):
    """|x| < 2^e: random, short, ties of every digit, the largest and the smallest."""
    top = np.nextafter(1.0, 0.0)
    v = list(rng.uniform(-1, 1, 300)) + [np.ldexp(m, -s) for m, s in
                                         zip(rng.choice([-1.0, 1.0], 100), rng.integers(1, 70, 100))]
    for beta in (8, 9):
        for s in range(1, 8):
            unit = 2.0 ** (-beta * s)
            v += [k * unit + h * unit for k in (-3, 0, 1, 2) for h in (-0.5, 0.5)]
            v += [0.5 + unit / 2, 0.5 - unit / 2, 1 - unit / 2, -1 + unit / 2, 1 - unit]
    v += [0.0, -0.0, top, -top, 0.5, -0.5, 2.0 ** -52, -(2.0 ** -53), 5e-324]
    return [float(np.ldexp(x, e)) for x in v if abs(x) < 1]


@pytest.mark.parametrize("beta,S", [(9, 6), (9, 7), (8, 7)])
def test_pair_digits(beta, S):
    rng = np.random.default_rng(beta * 10 + S)
    for x in values(rng, 0):
        d = pair_digits(float(np.ldexp(x, 3 * beta)), beta, S)
        assert abs(d[0]) <= 2 ** beta and all(abs(q) <= 2 ** (beta - 1) for q in d[1:]), (x, d)
        got = sum(Fraction(q) / Fraction(2) ** (beta * (s + 1)) for s, q in enumerate(d))
        assert abs(got - Fraction(x)) <= Fraction(1, 2 ** (beta * S + 1)), (x, d)


def test_pair_digits_are_not_the_rounding_one_by_one():
    """0.5 is 1, -128 in base 256 here; rounding digit by digit (kami_split_slices) gives 0, 128."""
    assert pair_digits(0.5 * 2 ** 16, 8, 7)[:2] == [1, -128]
    r = 0.5
    assert (round(r), round((r - round(r)) * 256)) == (0, 128)


def digit_word(x, E):
    scale = 1000 if E < -960 else -1000 if E > 960 else 0
    x, E = float(np.ldexp(x, scale)), E + scale
    h = (1023 + 22 + E) << 20 | 0x80000
    low_h = h - (32 << 20)
    high, low = double(h << 32), double(low_h << 32)
    t1 = x + high
    t2 = (x - (t1 - high)) + low
    fix = (0x80808080 - low_h) & 0xFFFFFFFF
    Y = (bits(t2) + ((((bits(t1) & 0xFFFFFFFF) + fix) & 0xFFFFFFFF) << 32 | 0x80808080)) & (2 ** 64 - 1)
    return Y ^ 0x8080808080808080


@pytest.mark.parametrize("E", [-1073, -1050, -1022, -961, -960, -1, 0, 1, 14, 960, 961, 1023, 1024])
def test_int8_digits_are_the_nearest(E):
    rng = np.random.default_rng(E + 2000)
    for x in values(rng, E):
        if not np.isfinite(x):
            continue
        word = digit_word(x, E)
        d = [((word >> (8 * b)) & 0xFF) - 256 * (((word >> (8 * b)) & 0xFF) >> 7) for b in range(8)]
        got = sum(q << (8 * b) for b, q in enumerate(d))
        assert got == round(Fraction(x) * Fraction(2) ** (62 - E)), (x, E)  # nearest, ties to even
