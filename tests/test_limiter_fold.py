"""The device's FP64 limiter folds the reference's halves; where that rounds alike.

The reference halves |f0 - f-1| and halves |c1 f0 + c2 f-1| twice before it adds
them and multiplies by |s0 + s1|.  The device forms D = |f0 - f-1| + |g| / 2 in
one fused multiply-add and |f - f0| - q D / 2 in another.  Halving is exact unless the
result is subnormal, so above 2^-1018 both give the same bits.  Below, the
device rounds once where the reference rounds up to four times: the subtracted terms
may differ by the reference's extra roundings, at most 3 units of 2^-1074 (two from
the halves of g and one from that of the difference, half a unit each and times
q <= 2), and where the values are still normal that may tip the roundings of the
excess and of the state, one spacing of the values each.
Both formulas are restated here (the oracle is the reference's), with fused
multiply-adds rounded from exact fractions.
"""
from fractions import Fraction

import numpy as np
import pytest

from oracle_lib import pdmu7

TINY = 2.0 ** -1074
PICK = (0, 0, 0, 1, 0, 0, 0)  # weights: the interpolant is the fourth value


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def folded(f_itp, fm1, f0, fp1, c1, c2):
    lo, hi = min(f0, fp1), max(f0, fp1)
    f = max(lo, min(f_itp, hi))
    d0, d1 = f0 - fm1, fp1 - f0
    q = 0.5 if d0 == 0.0 else (0.0 if np.signbit(d0) != np.signbit(d1) else 1.0)
    g = c1 * f0 + c2 * fm1
    D = fma(0.5, abs(g), abs(d0))
    t = max(0.0, fma(-q, D, abs(f - f0)))
    return f - float(np.copysign(t, d1))


def geometry(rng):
    """Face areas, volume and width, and the two terms the tables hold."""
    am, a, vol, dx = (float(x) for x in rng.uniform(0.5, 2.0, 4))
    q, e = vol / dx, 1.0 / 3.0
    return (am, a, vol, dx), (q - e * a) / (e * a), (e * am - q) / (e * a)


def samples(rng, scale):
    """Cells of one magnitude, some equal, zero or a few units apart."""
    x = rng.standard_normal(4) * scale
    kind = rng.integers(8)
    if kind == 0:
        x[2] = x[1]
    elif kind == 1:
        x[3] = x[2]
    elif kind == 2:
        x[rng.integers(4)] = rng.choice([0.0, -0.0])
    elif kind == 3:
        x[:] = x[0] + rng.integers(-4, 5, 4) * max(abs(x[0]) * 2.0 ** -52, TINY)
    return [float(v) for v in x]


def both(rng, scale):
    f_itp, fm1, f0, fp1 = samples(rng, scale)
    (am, a, vol, dx), c1, c2 = geometry(rng)
    fh = [0.0, 0.0, 0.0, f_itp, 0.0, 0.0, 0.0]
    ref = pdmu7(fh, [0.0, 0.0, fm1, f0, fp1, 0.0, 0.0], PICK, am, a, vol, dx)
    return ref, folded(f_itp, fm1, f0, fp1, c1, c2)


@pytest.mark.parametrize("exponent", [0, 300, -300, -900, -960])
def test_same_bits_where_no_half_is_subnormal(exponent):
    # differences of such values are multiples of 2^(exponent - 52), so no half is subnormal
    rng = np.random.default_rng(1000 + exponent)
    for _ in range(3000):
        ref, dev = both(rng, 2.0 ** exponent)
        assert ref == dev


@pytest.mark.parametrize("exponent", [-1020, -1040, -1060, -1070, -1073])
def test_a_few_units_apart_below(exponent):
    rng = np.random.default_rng(2000 - exponent)
    apart = 0
    for _ in range(3000):
        ref, dev = both(rng, 2.0 ** exponent)
        bound = 3 * Fraction(TINY) + 2 * Fraction(float(np.spacing(8 * 2.0 ** exponent)))
        assert abs(Fraction(ref) - Fraction(dev)) <= bound
        apart += ref != dev
    print("values apart:", apart, "of 3000")


def test_the_difference_exists():
    # f0 - f-1 = 3 units: its half, 1.5, rounds to 2 in the reference; g = 0
    unit = TINY
    fh = [0.0] * 3 + [20 * unit] + [0.0] * 3
    ref = pdmu7(fh, [0, 0, 0.0, 3 * unit, 40 * unit, 0, 0], PICK, 1 / 3, 1.0, 1 / 3, 1.0)
    dev = folded(20 * unit, 0.0, 3 * unit, 40 * unit, 0.0, 0.0)
    assert (ref / unit, dev / unit) == (7.0, 6.0)
