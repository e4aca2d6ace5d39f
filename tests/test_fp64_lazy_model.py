"""Exact model of the rescale's FP64 steps on limbs below 2^41 (th_device.h, ntt_arith.h).

reduce_u64_f64 takes the coefficient-domain last limb c < 2^61 to a residue of
small magnitude, the input of the forward transform, without corrections:
    r = fma(fma(-rint(ch 2^32 / q), q / 2^32, ch), 2^32, cl),  c = ch 2^32 + cl,
and the rescale's store forms (c - x) q_last^{-1} from the transform's output x
as it is (|x| < 9 q + 2^32: the input and at most 15 stages of 0.51 q). The same IEEE-754 operations with Python's floats, fused
multiply-adds rounded once from the exact rational value.
"""
from fractions import Fraction

import numpy as np
import pytest

from provenloop_amd.params import CHAIN_N32768_L8

# limb primes of the default chains, the largest of the path, and small ones
QS = sorted({q for q in [1099510054913, 1099508121601, 1099511480321, 1099510890497] + CHAIN_N32768_L8 if q < 1 << 41}
            | {2199023190017, 1073643521, 786433, 12289})


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def rint(x):
    return float(round(x))


def reduce_u64(c, q):
    ch, cl = float(c >> 32), float(c & 0xFFFFFFFF)
    quot = rint(ch * (4294967296.0 / float(q)))
    return fma(fma(-quot, float(q) / 4294967296.0, ch), 4294967296.0, cl)


def mulmod(x, w, wq, q):
    hi = x * w
    lo = fma(x, w, -hi)
    return fma(-rint(x * wq), q, hi) + lo


def mulmod_any(a, b, q):
    hi = a * b
    lo = fma(a, b, -hi)
    return fma(-rint(hi * (1.0 / q)), q, hi) + lo


def to_u64(x):
    """x + 2^52, mantissa bits."""
    return int(np.float64(x + 4503599627370496.0).view(np.uint64)) & 0xFFFFFFFFFFFFF


def from_u64(v):
    return float(np.uint64(v | 0x4330000000000000).view(np.float64)) - 4503599627370496.0


@pytest.mark.parametrize("q", QS)
def test_reduction_is_a_small_residue(q):
    rng = np.random.default_rng(q % 65521)
    edges = [0, 1, q - 1, q, 2 * q, (1 << 32) - 1, 1 << 32, (1 << 60) - 1, 1 << 60, (1 << 61) - 1]
    for t in range(1, 40):  # high words next to the ties of rint
        ch = ((2 * t + 1) * q) >> 33
        edges += [ch << 32, (ch << 32) | 0xFFFFFFFF, (ch + 1) << 32]
    for c in edges + [int(v) for v in rng.integers(0, 1 << 61, 2000, dtype=np.uint64)]:
        r = reduce_u64(c, q)
        assert r == int(r) and (int(r) - c) % q == 0
        assert abs(r) <= 0.76 * q + 4294967296.0  # 0.52 q from q = 2^21 on


@pytest.mark.parametrize("q", QS)
def test_store_from_the_raw_output(q):
    rng = np.random.default_rng(q % 65519)
    qd = float(q)
    top = 9 * q + (1 << 32)
    edges = [0, -1, q, -q, top, -top, 1 << 32, -(1 << 32)]
    for x in edges + [int(v) for v in rng.integers(-top, top + 1, 400)]:
        a, b, inv = (int(v) % q for v in rng.integers(0, 1 << 60, 3, dtype=np.uint64))
        c = mulmod_any(float(a), float(b), qd)
        assert (int(c) - a * b) % q == 0 and abs(c) <= 0.51 * qd
        r = mulmod(c - float(x), float(inv), float(inv) / qd, qd)
        r = r + qd if r < 0.0 else r
        assert to_u64(r) == (a * b - x) * inv % q


def test_conversions():
    for v in [0, 1, (1 << 41) - 1, (1 << 52) - 1, 1099510054912] + [int(v) for v in
                                                                   np.random.default_rng(1).integers(0, 1 << 52, 500)]:
        assert from_u64(v) == float(v) and to_u64(float(v)) == v
