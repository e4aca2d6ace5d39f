"""The work a user of this package has it do, as measurable cases.

Every case is a dict of plain values; `kind` names the path:

  token  one token of the encrypted LoRA path through a device-resident LoRA
         set (zero_moai.LoraSet): encrypt_pk per input, ct x pt per packed
         batch, rescale, batched decryption with segment sums, B on the GPU;
  ntt    raw batched negacyclic transforms of device-resident residues;
  calls  the drop-in module's per-call sequence of one layer: encrypt_pk,
         ct * numpy plaintext per packed batch, decrypt per product;
  batch  the same operations through the batched entry points, the slots left
         in device memory;
  keys   a session's set-up: keygen, keygen_public, and the key material out.

Sizes are those of bench.py, tests/ and provenloop_amd/params.py (Qwen2.5-1.5B
shape: 28 layers, hidden 1536, q and v, rank 16, N = 16384; Qwen2.5-7B shape:
hidden 3584, q, k, v and o, rank 32, N = 32768 on the 8-limb chain), or odd
generic ones.
"""
import ctypes
import math

import numpy as np
import torch

from provenloop_amd import _lib, params, tensafe_he, zero_moai

CHAINS = {
    8192: [1152921504606830593, 1099511480321, 1099510890497, 1152921504606601217],
    16384: [1152921504606748673, 1099510054913, 1099508121601, 1152921504606683137],
    32768: [1152921504606584833, 1099507695617, 1099506515969, 1152921504598720513],
}
COST_MAX = 896 * 32768 * 8  # residues of the largest listed case's products (per component)


def listed():
    return [
        # One encrypted delta, host floats in and out: what a user waits for
        # when a single adapter answers (bench.py --workload single).
        dict(name="delta", kind="token", n=16384, limbs=4, inputs=1, per_input=1, d=1536, rank=16, experts=0,
             rescale=True, sk_fused=False, host=True, ship=False),
        # The smallest degree with odd sizes, and the products taken out as
        # residues, as a server does that sends them back to its client.
        dict(name="delta_shipped", kind="token", n=8192, limbs=4, inputs=3, per_input=2, d=1001, rank=7, experts=0,
             rescale=True, sk_fused=False, host=True, ship=True),
        # A token of the 1.5B shape, inputs and deltas in HBM, one
        # synchronisation: the benchmark's step.
        dict(name="token", kind="token", n=16384, limbs=4, inputs=28, per_input=2, d=1536, rank=16, experts=0,
             rescale=True, sk_fused=False, host=False, ship=False),
        # The reference engine's own sequence for it: no rescale, CRT decryption.
        dict(name="token_unscaled", kind="token", n=16384, limbs=4, inputs=28, per_input=2, d=1536, rank=16,
             experts=0, rescale=False, sk_fused=False, host=False, ship=False),
        # One party holds the secret key: the shortcut, host arrays in and out.
        dict(name="token_sk_fused", kind="token", n=16384, limbs=4, inputs=28, per_input=2, d=1536, rank=16,
             experts=0, rescale=True, sk_fused=True, host=True, ship=False),
        # CryptoMOE: three experts a projection, new gates for the token.
        dict(name="token_moe", kind="token", n=16384, limbs=4, inputs=28, per_input=2, d=1536, rank=16, experts=3,
             rescale=True, sk_fused=False, host=False, ship=False),
        # A session-token of the 7B shape on the long chain (saturation serving).
        dict(name="session_7b", kind="token", n=32768, limbs=8, inputs=56, per_input=2, d=3584, rank=32, experts=0,
             rescale=True, sk_fused=False, host=False, ship=False),
        # The raw transforms in the microbenchmark's shape, forward ...
        dict(name="ntt_forward", kind="ntt", n=16384, limbs=4, count=64, inverse=False),
        # ... and inverse at the largest degree.
        dict(name="ntt_inverse", kind="ntt", n=32768, limbs=4, count=64, inverse=True),
        # One layer's q and v through the drop-in module, call by call, as the
        # reference's engine drives it.
        dict(name="calls_layer", kind="calls", n=16384, d=1536, rank=32),
        # A token's worth of ciphertexts through the batched entry points, with
        # full decoding to device memory (decrypt_to_gpu for a batch).
        dict(name="batch_ops", kind="batch", n=16384, inputs=28, per_input=4, d=1536, rescale=True),
        # What a new session pays once.
        dict(name="session_keys", kind="keys", n=16384),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 1e-9)))))


def draw(rng):
    kind = rng.choice(["token"] * 6 + ["ntt"] * 2 + ["calls", "batch", "batch", "keys"])
    n = rng.choice([8192, 16384, 32768])
    if kind == "keys":
        return dict(kind=kind, n=n, salt=rng.randrange(1 << 20))  # salt: another key pair
    if kind == "ntt":
        limbs = rng.randint(1, 4)
        return dict(kind=kind, n=n, limbs=limbs, count=_log_int(rng, 1, 256), inverse=rng.random() < 0.5)
    d = _log_int(rng, 512, 4096)
    if kind == "calls":
        return dict(kind=kind, n=n, d=d, rank=_log_int(rng, 1, 32))
    if kind == "batch":
        return dict(kind=kind, n=n, inputs=_log_int(rng, 1, 32), per_input=rng.randint(1, 6), d=d,
                    rescale=rng.random() < 0.5)
    case = dict(kind=kind, n=n, limbs=8 if n == 32768 and rng.random() < 0.5 else 4, inputs=_log_int(rng, 1, 32),
                per_input=rng.randint(1, 4), d=d, rank=_log_int(rng, 1, 64),
                experts=rng.choice([0, 0, 0, 2, 3, 4]), rescale=rng.random() < 0.8, sk_fused=rng.random() < 0.3,
                host=rng.random() < 0.5, ship=False)
    while case["inputs"] > 1 and _batches(case) * max(1, case["experts"]) * n * case["limbs"] > COST_MAX // 2:
        case["inputs"] -= 1
    return case


# ---------------------------------------------------------------- inputs
def _batches(case):
    cols = (case["n"] // 2) // case["d"]
    return case["inputs"] * case["per_input"] * -(-case["rank"] // cols)


def _chain(case):
    return params.CHAIN_N32768_L8 if case.get("limbs") == 8 else CHAINS[case["n"]]


def _context(case):
    return (tensafe_he.CkksContext(case["n"], moduli=params.CHAIN_N32768_L8) if case.get("limbs") == 8
            else tensafe_he.CkksContext(case["n"]))


def _d_outs(case):
    # q and o as wide as the input, k and v narrow (grouped-query attention)
    return [case["d"] if p % 2 == 0 else max(1, case["d"] // 6) for p in range(case["per_input"])]


def _token_data(case, seed):
    """Hidden states ~ 0.1 N(0, 1), adapters ~ 0.02 N(0, 1) as served f32 values, softmax gates."""
    rng = np.random.default_rng([seed, 1])
    k = max(1, case["experts"])
    d, r = case["d"], case["rank"]

    def f32(shape, s):
        return (rng.standard_normal(shape, dtype=np.float32) * np.float32(s)).astype(np.float64)

    hidden = f32((case["inputs"], d), 0.1)
    proj = []
    for i in range(case["inputs"]):
        for o in _d_outs(case):
            proj.append((i, f32((k, r, d), 0.02), f32((k, o, r), 0.02)))
    logits = rng.standard_normal((len(proj), k))
    g = np.exp(logits - logits.max(axis=1, keepdims=True))
    return hidden, proj, g / g.sum(axis=1, keepdims=True)


def _seeds(case, seed):
    return np.random.default_rng([seed, 2]).integers(0, 1 << 63, case["inputs"], dtype=np.uint64)


def _ntt_data(case, seed):
    rng = np.random.default_rng([seed, 3])
    q = _chain(case)[:case["limbs"]]
    return np.stack([rng.integers(0, m, (case["count"], case["n"]), dtype=np.uint64) for m in q], axis=1)


def _vectors(case, seed):
    """Replicated hidden states and packed plaintexts for the per-call and batched operations."""
    rng = np.random.default_rng([seed, 4])
    S, d = case["n"] // 2, case["d"]
    cols = S // d
    inputs = case.get("inputs", 1)
    h = [zero_moai.replicate(rng.standard_normal(d) * 0.1, S, d) for _ in range(inputs)]
    if case["kind"] == "calls":
        pts = zero_moai.pack_rows(rng.standard_normal((case["rank"], d)) * 0.02, S)
    else:
        pts = [zero_moai.pack_rows(rng.standard_normal((cols, d)) * 0.02, S)[0]
               for _ in range(inputs * case["per_input"])]
    return h, pts


# ---------------------------------------------------------------- the case protocol
def prepare(case, seed):
    st = {"case": case}
    ctx = st["ctx"] = _context(case)
    if case["kind"] == "keys":
        s = np.random.default_rng([seed, case.get("salt", 0), 5]).integers(0, 1 << 62, 2)
        st["seeds"] = (int(s[0]), int(s[1]))
        return st
    if case["kind"] == "ntt":
        st["src"] = torch.from_numpy(_ntt_data(case, seed).view(np.int64)).cuda()
        st["out"] = torch.empty_like(st["src"])
        p = ctypes.c_void_p()
        _lib.check(_lib.load().th_ctx_stream(ctx._h, ctypes.byref(p)))
        st["stream"] = torch.cuda.ExternalStream(p.value)
        return st
    st["sk"] = ctx.keygen(seed=2 * seed + 1)
    st["pk"] = ctx.keygen_public(st["sk"], seed=2 * seed + 2)
    if case["kind"] == "token":
        hidden, proj, gates = _token_data(case, seed)
        if case["experts"]:
            st["set"] = zero_moai.LoraSet(ctx, case["inputs"], proj, gates=np.full_like(gates, 1.0 / gates.shape[1]))
            st["gates"] = gates
        else:
            st["set"] = zero_moai.LoraSet(ctx, case["inputs"], [(i, a[0], b[0]) for i, a, b in proj])
        st["seeds"] = _seeds(case, seed)
        if case["host"]:
            st["hidden"] = hidden
        else:
            st["hidden"] = torch.from_numpy(hidden).cuda()
            st["deltas"] = torch.empty(st["set"].n_deltas, dtype=torch.float64, device="cuda")
        return st
    h, pts = _vectors(case, seed)
    st["h"] = h
    if case["kind"] == "calls":
        st["pts"] = pts
        st["seed"] = int(seed) * 7 + 3
    else:
        st["pts"] = [ctx.encode_to_ntt(p) for p in pts]
        st["seeds"] = [int(s) for s in _seeds(case, seed)]
        st["slots"] = torch.empty((len(pts), ctx.num_slots), dtype=torch.float64, device="cuda")
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    if case["kind"] == "keys":
        sk = ctx.keygen(seed=st["seeds"][0])
        pk = ctx.keygen_public(sk, seed=st["seeds"][1])
        return {"pk": np.frombuffer(pk.to_bytes(), np.int64), "sk": ctx.sk_download(sk).view(np.int64)}
    if case["kind"] == "ntt":
        lib = _lib.load()
        fn = lib.th_ntt_inverse_batch if case["inverse"] else lib.th_ntt_forward_batch
        with torch.cuda.stream(st["stream"]):  # the input stays for the caller: the transform is in place
            st["out"].copy_(st["src"])
        _lib.check(fn(ctx._h, st["out"].data_ptr(), case["count"], case["limbs"], 1))
        return st["out"]
    sk, pk = st["sk"], st["pk"]
    if case["kind"] == "token":
        ls = st["set"]
        if case["experts"]:
            ls.set_gates(st["gates"])
        if case["host"]:
            out = {"deltas": ls.deltas(pk, sk, st["hidden"], st["seeds"], rescale=case["rescale"],
                                       sk_fused=case["sk_fused"])}
            out["deltas"] = np.concatenate(out["deltas"])
        else:
            ls.deltas_device(pk, sk, st["hidden"].data_ptr(), st["seeds"], st["deltas"].data_ptr(),
                             rescale=case["rescale"], sk_fused=case["sk_fused"])
            ctx.sync()
            out = {"deltas": st["deltas"]}
        if case["ship"]:
            out["products"] = [np.frombuffer(ls.ciphertext("product", b).to_bytes()[8:], np.int64)
                               for b in range(ls.n_batches)]
        return out
    if case["kind"] == "calls":
        ct = ctx.encrypt_pk(st["h"][0], pk, seed=st["seed"])
        return {"slots": [ctx.decrypt(ct * p, sk) for p in st["pts"]]}
    cts = ctx.encrypt_pk_batch(st["h"], pk, st["seeds"])
    prods = ctx.ct_pt_mul_ntt_batch([cts[j // case["per_input"]] for j in range(len(st["pts"]))], st["pts"])
    if case["rescale"]:
        prods = ctx.rescale_batch(prods)
    ctx.batch_decrypt_to_device(prods, sk, st["slots"].data_ptr())
    return {"slots": st["slots"]}


def work(case):
    """Bytes: keys, plaintexts and inputs in, ciphertexts formed and results out, once each. Operations: one modular
    product and two sums a butterfly, and the encoder's and decoder's FFTs."""
    n = case["n"]
    L = case.get("limbs", 4)
    P, fly, fft = 8 * n, 3 * (n / 2) * math.log2(n), 5 * n * math.log2(n)
    if case["kind"] == "ntt":
        t = case["count"] * L
        return {"bytes": 2 * P * t, "flops": fly * t}
    if case["kind"] == "keys":
        return {"bytes": 3 * L * P, "flops": 3 * L * fly}
    if case["kind"] == "calls":
        nb = -(-case["rank"] // ((n // 2) // case["d"]))
        return {"bytes": 2 * L * P + nb * (2 * L * P) + 8 * (n // 2) * (1 + 2 * nb),
                "flops": 3 * L * fly + fft + nb * (L * fly + 2 * fly + 2 * fft)}
    if case["kind"] == "batch":
        ni, nb = case["inputs"], case["inputs"] * case["per_input"]
        tr = (2 + 2 * (L - 1) + 1) if case["rescale"] else 2
        return {"bytes": 2 * L * P + ni * 2 * L * P + nb * (L * P + 2 * L * P + 8 * (n // 2)),
                "flops": ni * (3 * L * fly + fft) + nb * (tr * fly + fft)}
    ni, nb, k = case["inputs"], _batches(case), max(1, case["experts"])
    outs = sum(_d_outs(case)) * ni
    io = 8 * (ni * case["d"] + outs + outs * case["rank"] * k)
    if case["sk_fused"]:
        le = 2 if case["rescale"] else 2
        by, tr = le * 2 * P + nb * 2 * P, ni * 3 * le + nb * (4 if case["rescale"] else 2)
    elif case["rescale"]:
        by = 2 * L * P + ni * 2 * L * P + nb * (L * P + 2 * (L - 1) * P)
        tr = ni * 3 * L + nb * (2 + 2 * (L - 1) + 1)
    else:
        by, tr = 2 * L * P + ni * 2 * L * P + nb * (L * P + 2 * L * P), ni * 3 * L + nb * 2
    fl = tr * fly + ni * fft + 2 * outs * case["rank"]
    if case["experts"]:
        by += nb * k * 8 * (n // 2) + nb * L * P
        fl += nb * k * fft + nb * L * fly
    return {"bytes": by + io, "flops": fl}


def tolerance(case):
    # Residues, keys and fully decoded slots equal the reference's bit for bit.
    # The segment sums behind the deltas may be added in another order (1.3e-15
    # measured between the set's sums and the oracle's decode-then-sum).
    return {"rel": 6e-15} if case["kind"] == "token" else "exact"


# ---------------------------------------------------------------- plain evaluation
def _mulmod(a, b, q):
    """a * b mod q for uint64 arrays below q < 2^60: quotient from 64-bit-mantissa products, off by at most one."""
    quot = (a.astype(np.longdouble) * b.astype(np.longdouble) / np.longdouble(q)).astype(np.uint64)
    r = (a * b - quot * np.uint64(q)).view(np.int64)
    r = np.where(r < 0, r + np.int64(q), r)
    return np.where(r >= q, r - np.int64(q), r).astype(np.uint64)


def _transform(x, q, n, inverse):
    """Negacyclic transform of x [count, n] mod q over the powers of psi = the first g^((q-1)/2n) of order 2n, in the
    bit-reversed order of the reference."""
    logn = n.bit_length() - 1
    g = 2
    while pow(psi := pow(g, (q - 1) // (2 * n), q), n, q) != q - 1:
        g += 1
    if inverse:
        psi = pow(psi, q - 2, q)
    w, p = np.zeros(n, np.uint64), 1
    for i in range(n):
        w[int(format(i, "0%db" % logn)[::-1], 2)] = p
        p = p * psi % q
    x, m64 = x.copy(), np.uint64(q)
    for s in (range(logn - 1, -1, -1) if inverse else range(logn)):
        m = 1 << s
        y = x.reshape(x.shape[0], m, 2, n // (2 * m))
        t = w[m:2 * m].reshape(1, m, 1)
        if not inverse:
            u, v = y[:, :, 0].copy(), _mulmod(y[:, :, 1], np.broadcast_to(t, y[:, :, 1].shape), q)
            y[:, :, 0], y[:, :, 1] = (u + v) % m64, (u + m64 - v) % m64
        else:
            u, v = y[:, :, 0].copy(), y[:, :, 1].copy()
            y[:, :, 0] = (u + v) % m64
            y[:, :, 1] = _mulmod((u + m64 - v) % m64, np.broadcast_to(t, v.shape), q)
    if inverse:
        x = _mulmod(x, np.broadcast_to(np.uint64(pow(n, q - 2, q)), x.shape), q)
    return x


def exact(case, seed):
    if case["kind"] == "keys":
        return None  # drawn, not computed
    if case.get("rescale") and case["kind"] != "ntt":
        # The chains end in a 60-bit prime, so a rescaled product has scale
        # 2^80 / 2^60 and these values lie below the scheme's own rounding:
        # what comes back is fixed by the drawn randomness, not by the inputs.
        return None
    if case["kind"] == "ntt":
        if case["count"] * case["limbs"] * case["n"] > 1 << 23:
            return None
        x = _ntt_data(case, seed)
        for i, q in enumerate(_chain(case)[:case["limbs"]]):
            x[:, i] = _transform(x[:, i], q, case["n"], case["inverse"])
        return x.view(np.int64)
    if case["kind"] == "token":
        hidden, proj, gates = _token_data(case, seed)
        if not case["experts"]:
            gates = np.ones((len(proj), 1))
        out = []
        for (i, a, b), g in zip(proj, gates):
            inter = sum(g[x] * (a[x] @ hidden[i]) for x in range(len(g)))
            out.append(sum(g[x] * b[x] for x in range(len(g))) @ inter)
        return {"deltas": np.concatenate(out)}
    h, pts = _vectors(case, seed)
    per = len(pts) if case["kind"] == "calls" else case["per_input"]
    slots = [h[j // per] * p for j, p in enumerate(pts)]
    return {"slots": slots if case["kind"] == "calls" else np.stack(slots)}
