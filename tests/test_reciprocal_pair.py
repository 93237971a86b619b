"""The reciprocal pair behind the FP64 sweeps' division (reciprocal_pair in csrc/thomas.cpp):
where it returns true, RN(a*hi + RN(a*lo)) has to be the correctly rounded a/d for every
numerator a; where it finds no such pair (about one odd divisor in a thousand) lo is NaN.

Checked with exact rational arithmetic on the numerators whose quotient lies closest to the
midpoint of two neighbouring doubles (the only ones that can fail; they are solved for, A*2^k =
J mod D), on random ones, and on denominators as the Thomas recursion makes them.  No
tolerance: the two roundings agree or the test fails."""
import ctypes
import math
import os
import random
from fractions import Fraction

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "biofvm-b_amd", "lib", "libbiofvmb.so")


@pytest.fixture(scope="module")
def pair():
    import biofvmb._lib as L
    fn = ctypes.CDLL(L.LIB_PATH)["_ZN5bfvmb15reciprocal_pairEdPdS0_"]
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.c_double, ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_double)]

    def call(d):
        hi, lo = ctypes.c_double(), ctypes.c_double()
        ok = fn(d, ctypes.byref(hi), ctypes.byref(lo))
        return ok, hi.value, lo.value
    return call


def _rn(q):
    """Nearest double of a rational, ties to even (Fraction's true division of integers)."""
    return q.numerator / q.denominator


def _divide(a, hi, lo):
    t = _rn(Fraction(a) * Fraction(lo))
    return _rn(Fraction(a) * Fraction(hi) + Fraction(t))


def _numerators(d, rng, jmax=41):
    D = int(math.ldexp(math.frexp(d)[0], 53))
    out = [rng.randrange(1 << 52, 1 << 53) for _ in range(20)] + [1 << 52, (1 << 53) - 1]
    if D & 1:
        for k in (53, 54):
            inv = pow(pow(2, k, D), -1, D)
            for J in range(-jmax, jmax + 1):
                a = inv * J % D
                out += [x for x in (a, a + D) if 1 << 52 <= x < 1 << 53]
    return out


def test_random_divisors(pair):
    rng = random.Random(5)
    moved = refused = 0
    for _ in range(1200):
        d = math.ldexp(rng.randrange(1 << 52, 1 << 53) | 1, -52 + rng.randrange(0, 8))
        ok, hi, lo = pair(d)
        assert hi == 1.0 / d
        lo0 = _rn(1 / Fraction(d) - Fraction(hi))
        if not ok:
            assert np.isnan(lo)
            assert any(_divide(float(a), hi, lo0) != a / d for a in _numerators(d, rng))
            refused += 1
            continue
        moved += lo != lo0
        for a in _numerators(d, rng):
            x = math.ldexp(a, rng.randrange(-950, 900))
            assert _divide(x, hi, lo) == x / d, (d, a)
    assert moved > 0 and refused < 12


def test_known_failing_divisors_are_adjusted(pair):
    """Divisors whose nearest pair misrounds some numerator (found by the same search) come back
    with a pair that does not, or refused."""
    rng = random.Random(9)
    found = 0
    while found < 12:
        d = math.ldexp(rng.randrange(1 << 52, 1 << 53) | 1, -52)
        hi0 = 1.0 / d
        lo0 = _rn(1 / Fraction(d) - Fraction(hi0))
        num = _numerators(d, rng, jmax=3)
        if all(_divide(float(a), hi0, lo0) == a / d for a in num):
            continue
        found += 1
        ok, hi, lo = pair(d)
        assert not ok or lo != lo0
        for a in _numerators(d, rng) if ok else ():
            assert _divide(float(a), hi, lo) == a / d


@pytest.mark.parametrize("D,dt,dx,n", [(1e5, 0.01, 20.0, 400), (1e3, 0.01, 20.0, 60), (5e4, 1.0, 20.0, 120)])
def test_thomas_denominators(pair, D, dt, dx, n):
    c1 = D * dt / dx / dx
    den, seen, rng = 1.0 + c1 + 0.001, set(), random.Random(1)
    for _ in range(n):
        if den not in seen:
            seen.add(den)
            ok, hi, lo = pair(den)
            for a in _numerators(den, rng, jmax=9) if ok else ():
                assert _divide(float(a), hi, lo) == a / den
        den = (1.0 + 2 * c1 + 0.001) - c1 * c1 / den


def test_powers_of_two_and_refused(pair):
    for d in (1.0, 2.0, 1.5, 6.0):
        ok, hi, lo = pair(d)
        assert ok and all(_divide(float(a), hi, lo) == a / d for a in _numerators(d, random.Random(2)))
    for d in (0.0, -1.0, float("inf"), float("nan"), 1e-300, 1e300):
        ok, _, lo = pair(d)
        assert not ok and np.isnan(lo)
