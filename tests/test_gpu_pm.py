"""Transforms on the two arithmetics above 2^41, at their edges, against the oracle.

Chains whose large primes are all 2^60 - c (c < 2^26) fold products at bit 60;
any other large prime takes the whole chain to Shoup products. Values at the
residues' edges, one prime with c close to 2^26, on the whole-polynomial and
the split kernels.
"""
import numpy as np
import pytest

from oracle import oracle as orc
from provenloop_amd import tensafe_he

pytestmark = pytest.mark.gpu


def _is_prime(n):
    d, s = n - 1, 0
    while d % 2 == 0:
        d, s = d // 2, s + 1
    for a in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37):
        x = pow(a, d, n)
        if x in (1, n - 1):
            continue
        for _ in range(s - 1):
            x = x * x % n
            if x == n - 1:
                break
        else:
            return False
    return True


def _prime_from(start, n, step):
    q = start - (start - 1) % (2 * n)
    if step > 0 and q <= start:
        q += 2 * n
    while not _is_prime(q):
        q += step * 2 * n
    return q


def _chain(kind, n):
    top, edge = 1 << 60, (1 << 60) - (1 << 26)
    if kind == "pm":  # c small, c close to 2^26, and a prime of the fp64 path
        q = [_prime_from(top - 1, n, -1), _prime_from(edge, n, 1), orc.default_chain(16384)[1]]
        assert edge < q[1] < edge + (1 << 24)
    else:  # just outside the folding range on both sides, and the largest accepted
        q = [_prime_from(edge, n, -1), _prime_from(top, n, 1), _prime_from((1 << 61) - 1, n, -1),
             orc.default_chain(16384)[1]]
    return q


@pytest.mark.parametrize("kind", ["pm", "int"])
@pytest.mark.parametrize("n,polys", [(1024, 2), (8192, 1), (16384, 40), (32768, 2)])
def test_transforms_at_the_edges(kind, n, polys):
    q = _chain(kind, n)
    ctx = tensafe_he.CkksContext(n, moduli=q)
    rng = np.random.default_rng(n)
    x = np.stack([rng.integers(0, m, (polys, n), dtype=np.uint64) for m in q], axis=1)
    m1 = np.array(q, np.uint64)[:, None] - np.uint64(1)
    x[0] = m1  # every residue q - 1
    x[-1, :, ::2] = m1
    x[-1, :, 1::3] = 0
    fwd, inv = ctx.ntt_forward(x), ctx.ntt_inverse(x)
    for p in {0, polys // 2, polys - 1}:
        for l, m in enumerate(q):
            assert np.array_equal(fwd[p, l], orc.ntt_forward(x[p:p + 1, l], m)[0]), (p, l)
            assert np.array_equal(inv[p, l], orc.ntt_inverse(x[p:p + 1, l], m)[0]), (p, l)


@pytest.mark.parametrize("kind", ["pm", "int"])
def test_ciphertext_operations(kind):
    """encrypt_pk, ct x pt, rescale and decryption on both kinds of chain."""
    n = 8192
    q = _chain(kind, n)
    eng, ref = tensafe_he.CkksContext(n, moduli=q), orc.Context(n, moduli=q)
    sk, rsk = eng.keygen(seed=1), ref.keygen(1)
    pk, rpk = eng.keygen_public(sk, seed=2), ref.keygen_public(rsk, 2)
    rng = np.random.default_rng(3)
    v, w = rng.standard_normal(n // 2) * 1e3, rng.standard_normal(n // 2)
    ct, rct = eng.encrypt_pk(v, pk, seed=4), ref.encrypt_pk(v, rpk, 4)
    prod, rprod = ct * w, ref.ct_pt_mul(rct, w)
    res, rres = eng.rescale(prod), ref.rescale(rprod)
    for got, exp in ((ct, rct), (prod, rprod), (res, rres)):
        assert all(np.array_equal(a, b) for a, b in zip(eng.ct_download(got), ref.ct_data(exp)))
        assert np.array_equal(eng.decrypt(got, sk), ref.decrypt(exp, rsk))


@pytest.mark.parametrize("n,polys", [(8192, 341), (8192, 342), (16384, 171), (32768, 85), (32768, 86)])
def test_inverse_batches_around_64_mib(n, polys):
    """Larger batches take instances of their own from 64 MiB of residues on (3 limbs each)."""
    q = _chain("pm", n)
    ctx = tensafe_he.CkksContext(n, moduli=q)
    rng = np.random.default_rng(polys)
    x = np.stack([rng.integers(0, m, (polys, n), dtype=np.uint64) for m in q], axis=1)
    x[0] = x[-1] = np.array(q, np.uint64)[:, None] - np.uint64(1)
    inv = ctx.ntt_inverse(x)
    for p in (0, polys // 2, polys - 2, polys - 1):
        for l, m in enumerate(q):
            assert np.array_equal(inv[p, l], orc.ntt_inverse(x[p:p + 1, l], m)[0]), (p, l)
