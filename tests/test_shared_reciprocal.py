"""The shared-reciprocal pair term (csrc/nbody_terms.hpp) rounds as IEEE does.

Its quotients are q = q0 + (n - d q0) r with one reciprocal r per divisor.  That is n/d
correctly rounded for the double r nearest to 1/d, and for the other neighbour too where
1/d is all but a tie -- except for divisors 2 - u 2^-52 with a small odd u, where a few
numerators need the nearer one.  Both sides are enumerated here with the numerators whose
quotients lie closest to a rounding boundary.  Exact rational arithmetic, no GPU.
"""
import math
import random
from fractions import Fraction as F

import pytest

ULP = F(1, 2**53)  # of numbers in [1/2, 1)


def rn(x):
    """x rounded to the nearest double, ties to even (normal range)."""
    if x == 0:
        return F(0)
    e = x.numerator.bit_length() - x.denominator.bit_length()
    if abs(x) < F(2)**e:
        e -= 1
    u = F(2)**(e - 52)
    k = x / u
    f = math.floor(k)
    d = k - f
    if d > F(1, 2) or (d == F(1, 2) and f % 2):
        f += 1
    return f * u


def quotient(n, d, r):
    q0 = rn(n * r)
    return rn(rn(n - d * q0) * r + q0)


def near_reciprocals(d):
    """The doubles within (1/2 + 2^-35) ulp of 1/d, d in (1, 2)."""
    k = math.floor(1 / d / ULP)
    return [c * ULP for c in (k, k + 1) if abs(c * ULP - 1 / d) <= (F(1, 2) + F(1, 2**35)) * ULP]


def hard_numerators(B):
    """53-bit integers A < B for which A / B is within j / (B 2^54), j <= 3, of the middle of
    two doubles."""
    inv = pow(2**54, -1, B)
    out = []
    for j in (1, 2, 3):
        for s in (j, -j):
            A = s * inv % B
            if A >= 2**52 and ((A * 2**54 - s) // B) % 2:
                out.append(A)
    return out


def pairs(us):
    for u in us:
        B = 2**53 - u
        tops = [2**53 - 1 - k for k in range(min(u, 3))]  # numerators above the divisor
        for A in hard_numerators(B) + tops:
            yield F(A, 2**52), F(B, 2**52)


@pytest.mark.parametrize("us", [range(1, 2048, 2), range(2**21 - 1999, 2**21, 2),
                                range(2**52 - 1999, 2**52, 2), range(1, 2**52, 2**42 + 2)])
def test_hard_quotients_with_the_nearest_reciprocal(us):
    for n, d in pairs(us):
        assert quotient(n, d, rn(1 / d)) == rn(n / d)


def test_the_other_neighbour_matters_just_below_two_only():
    wrong = {}
    for n, d in pairs(range(1, 4096, 2)):
        for r in near_reciprocals(d):
            if quotient(n, d, r) != rn(n / d):
                wrong.setdefault(2**53 - int(d * 2**52), []).append(r)
    # a wrong neighbour exists where the tie is closer than 2^-35 ulp: u^2 2^-54 < 2^-35
    assert all(u * u < 2**19 for u in wrong) and max(map(len, wrong.values())) <= 3
    assert sum(map(len, wrong.values())) < 2**11


def isqrt_rn(s):
    """The correctly rounded square root of a double s in [1, 4)."""
    n = s * 2**210
    k = math.isqrt(int(n))
    x = F(2 * k + (1 if k * k != n else 0), 2**106)  # sticky bit
    return rn(x)


def test_whole_term_at_random_separations():
    rng = random.Random(7)
    for _ in range(400):
        s = F(rng.randrange(2**52, 2**54), 2**52)
        n = F(rng.randrange(2**52, 2**53) * rng.choice((-1, 1)), 2**rng.randrange(50, 56))
        root = F(math.isqrt(int(F(2**200) / s)), 2**100)
        y = rn(root * (1 + F(rng.randrange(-2**20, 2**20), 2**44)))  # rsq off by up to 2^-24
        g, h = rn(s * y), rn(y / 2)
        r0 = rn(F(1, 2) - h * g)
        g = rn(g + g * r0)
        d = rn(s - g * g)
        h = rn(h + h * r0)
        g = rn(g + d * h)
        d = rn(s - g * g)
        dist = rn(g + d * h)
        assert dist == isqrt_rn(s)
        den = rn(dist * s)
        y1 = rn(h + h)
        r = rn(rn(y1 * y1) * y1)
        r = rn(r + r * rn(1 - den * r))
        # r's distance from 1/den in ulps (the unit in its last place)
        u = F(2)**(math.frexp(float(r))[1] - 53)
        assert abs(r - 1 / den) <= (F(1, 2) + F(1, 2**35)) * u
        assert quotient(n, den, r) == rn(n / den)
