"""Exact model of the products modulo q = 2^60 - c (th_device.h, pm path).

Repeats pm_fold, pm_mul_fixed, pm_mul, pm_canon, the encryption's signed
operands and the butterflies of PmArith with Python integers, every step held
to the width of its register, and checks the bounds that the transforms rely
on: a product by a fixed operand below 2.5q for any 64-bit value, a general
product below 4q for a < 2^62, no forward value at 16q over a pass of four
stages, and no inverse value past 8q between passes.
"""
import numpy as np
import pytest

from provenloop_amd.params import CHAIN_N32768_L8

M32, M64, M30, M28 = (1 << 32) - 1, (1 << 64) - 1, (1 << 30) - 1, (1 << 28) - 1
# the 60-bit primes of the default chains, and the ends of the path's range
# (the bounds hold for any odd q in it)
QS = [1152921504606748673, 1152921504606683137, 1152921504606830593, 1152921504606601217,
      CHAIN_N32768_L8[0], CHAIN_N32768_L8[-1], (1 << 60) - 1, (1 << 60) - (1 << 26) + 1]


def u64(v):
    assert 0 <= v <= M64
    return v


def u32(v):
    assert 0 <= v <= M32
    return v


def fold(x, c):
    return u64((x >> 60) * c + (x & ((1 << 60) - 1)))


def canon(x, q, c):
    r = fold(x, c)
    return r - q if r >= q else r


def tw(w, q):
    v = (w << 32) % q
    return w & M30, w >> 30, v & M30, v >> 30


def mul_fixed(x, t, c):
    wl, wh, vl, vh = t
    x0, x1 = x & M32, x >> 32
    ab = u64(u64(x0 * wl) + x1 * vl)
    cd = u64(u64(x0 * wh) + x1 * vh)
    top = u32(cd >> 31)
    d = u64(((cd & 0x7fffffff) << 30) + ab)
    h = u32(top + (d >> 61))
    return u64(h * 2 * c + (d & ((1 << 61) - 1)))


def mul(a, b, c):
    a0, a1, b0, b1 = a & M30, u32(a >> 30), b & M30, b >> 30
    mid = u64(a1 * b0 + a0 * b1)
    e = u64(a1 * b1 + (mid >> 30))
    r = u64(((mid & M30) << 30) + a0 * b0 + (e & M32) * c)
    y = u64(u32(e >> 32) * c)
    return u64(r + ((y & M28) << 32) + u32(y >> 28) * c)


def values(q, top, rng, n=60):
    edge = [0, 1, q - 1, q, q + 1, 2 * q, 4 * q - 1, (1 << 60) - 1, 1 << 60, (1 << 32) - 1, 0xffffffff00000000, top - 1]
    return [v % top for v in edge] + [int(v) % top for v in rng.integers(0, 1 << 64, n, dtype=np.uint64)]


@pytest.mark.parametrize("q", QS)
def test_products_and_folds(q):
    c = (1 << 60) - q
    rng = np.random.default_rng(c % 65521)
    for x in values(q, 1 << 64, rng, 200):
        assert fold(x, c) % q == x % q and fold(x, c) < q + 16 * c
        assert canon(x, q, c) == x % q
        e = x - (1 << 64) if x >> 63 else x  # the same bits as a signed value
        s = fold(x ^ (1 << 63), c)
        assert (s - 8 * c) % q == e % q and s < q + 16 * c
    for w in values(q, q, rng):
        for x in values(q, 1 << 64, rng):
            r = mul_fixed(x, tw(w, q), c)
            assert r % q == x * w % q and 2 * r < 5 * q
        for a in values(q, 1 << 62, rng):
            r = mul(a, w, c)
            assert r % q == a * w % q and r < 4 * q
    # the encryption's m + e0: two folds and q - 16 c
    assert 2 * (q + 16 * c) + q - 16 * c <= 4 * q


@pytest.mark.parametrize("q", QS)
def test_forward_bounds(q):
    """Four stages from a folded first stage: X grows by at most 3q a stage and stays below 16q."""
    c = (1 << 60) - q
    bound = 4 * q  # as loaded, nothing folded in the first pass
    for _ in range(4):
        bound += 3 * q
    assert bound <= 1 << 64
    for _ in range(3):  # later passes: any 64-bit value in, the first stage folds
        bound = q + 16 * c
        for _ in range(4):
            bound += 3 * q
        assert bound <= 1 << 64


@pytest.mark.parametrize("rb0,ns", [(0, 4), (0, 3), (1, 3), (2, 2), (0, 2), (1, 2), (3, 1), (2, 1)])
def test_inverse_plan(rb0, ns):
    """InvPlan in quarters of q: differences stay in (0, 16q), values between passes at or below 8q."""
    bound = [32] * 16
    for s in range(ns):
        for k in range(16):
            m = 1 << (rb0 + s)
            if k & m:
                continue
            add = 12 if bound[k | m] <= 12 else 32
            assert bound[k | m] <= add and bound[k] + add <= 64
            total = bound[k] + bound[k | m]
            assert total <= 64
            bound[k], bound[k | m] = (5 if total > 32 else total), 10
    assert max(bound) <= 32
