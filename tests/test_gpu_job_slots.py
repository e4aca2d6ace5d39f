"""Short job lists stay in a ring of pinned slots that the kernels read.

More operations than the ring has slots (4096 lists of up to 256 bytes), so
slots are handed out again after a lap: the running sum of a ciphertext with
itself must still be exact, and lists on both sides of the slot size (a batch
of one product, and one of many) give the same residues. That a lap waits for
what is queued before a slot is rewritten is tested on the host
(test_launch_rules.py): calls come too slowly to overtake the GPU by a lap.
"""
import numpy as np
import pytest

from provenloop_amd import tensafe_he

pytestmark = pytest.mark.gpu


def test_more_operations_than_slots():
    n, laps = 8192, 4300
    eng = tensafe_he.CkksContext(n)
    q = np.array([1152921504606830593, 1099511480321, 1099510890497, 1152921504606601217], dtype=object)
    rng = np.random.default_rng(2)
    c = np.stack([rng.integers(0, int(m), n, dtype=np.uint64) for m in q])
    step = eng.ct_upload(c, c, 2.0**40)
    acc = eng.ct_upload(np.zeros_like(c), np.zeros_like(c), 2.0**40)
    for _ in range(laps):
        acc = acc + step
    exp = (c.astype(object) * laps % q[:, None]).astype(np.uint64)
    for got in eng.ct_download(acc):
        assert np.array_equal(got, exp)


@pytest.mark.parametrize("count", [1, 9, 10, 13, 40])
def test_lists_on_both_sides_of_a_slot(count):
    n = 8192
    eng = tensafe_he.CkksContext(n)
    sk = eng.keygen(seed=1)
    pk = eng.keygen_public(sk, seed=2)
    rng = np.random.default_rng(count)
    ct = eng.encrypt_pk(rng.standard_normal(n // 2), pk, seed=3)
    pts = [eng.encode_to_ntt(rng.standard_normal(n // 2)) for _ in range(count)]
    batch = eng.rescale_batch(eng.ct_pt_mul_ntt_batch([ct] * count, pts))
    for i in {0, count // 2, count - 1}:
        one = eng.rescale(eng.ct_pt_mul_ntt(ct, pts[i]))
        assert all(np.array_equal(a, b) for a, b in zip(eng.ct_download(one), eng.ct_download(batch[i])))
        assert np.array_equal(eng.decrypt(one, sk), eng.decrypt(batch[i], sk))
