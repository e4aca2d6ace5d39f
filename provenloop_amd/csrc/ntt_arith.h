// Butterfly arithmetic and load-side operations shared by the NTT kernels.
//
// Three exact modular-multiply policies (with_arith: by the limb's prime, PmArith
// or IntArith by the chain, LimbTable). The transform kernels are templates of
// the larger one, compiled once for each:
//  PmArith   - q = 2^60 - c: products folded at bit 60. Values run up to 16q
//              (below 2^64): forward butterflies add at most 3q, so only the
//              first stage of a register pass folds its upper inputs; inverse
//              sums are folded where they could pass 8q (InvPlan).
//  IntArith  - 64-bit Shoup products with an approximate quotient (at most
//              2 short) and lazy ranges [0, 8q) forward, [0, 4q) inverse;
//              q < 2^61 so that 8q fits in 64 bits.
//  Fp64Arith - q < 2^41: exact products from one FMA split and a quotient
//              rounded from x * (w / q); values are exact integers in doubles.
// Both end on the canonical residue, so transforms are bit-identical to the
// reference's u128 Barrett NTT (tensafe-he-core/src/ntt.rs:79-141).
// raw()/unraw() carry a policy's intermediate values through global memory
// between the two kernels of a split transform (u64 lazy residues, or the
// bit pattern of the double).
#pragma once
#include <type_traits>

#include "th_internal.h"

namespace th {

// ------------------------------------------------------------------ arithmetic policies
struct IntArith {
  using V = uint64_t;
  using Tw = ShoupTw;
  uint64_t q, two_q, four_q;
  __device__ IntArith(const LimbConst& c) : q(c.q), two_q(c.two_q), four_q(2 * c.two_q) {}
  // 2^64 - 4q, the forward butterfly's csub_n addend (the same value at every
  // call, so the compiler keeps one copy)
  __device__ __forceinline__ uint64_t n4q() const { return opaque_u64(0 - four_q); }
  __device__ __forceinline__ V load(uint64_t x) const { return x; }
  // forward CT butterfly, inputs/outputs in [0, 8q): X < 4q, T < 4q
  __device__ __forceinline__ void fwd(V& a, V& b, const Tw& t, bool) const {
    const uint64_t X = csub_n(a, four_q, n4q());
    const uint64_t T = shoup_approx(b, t.w, t.ws, q);
    a = X + T;
    b = X + four_q - T;
  }
  // inverse GS butterfly, inputs/outputs in [0, 4q)
  __device__ __forceinline__ void inv(V& a, V& b, const Tw& t, bool, bool) const {
    const uint64_t X = a, Y = b;
    a = csub_n(X + Y, four_q, n4q());
    b = shoup_approx(X + four_q - Y, t.w, t.ws, q);
  }
  // last inverse stage with N^{-1} folded in; canonical outputs
  __device__ __forceinline__ void inv_last(V& a, V& b, const LimbConst& c) const {
    const uint64_t X = a, Y = b;
    a = csub(csub(shoup_approx(X + Y, c.n_inv, c.n_inv_s, q), two_q), q);
    b = csub(csub(shoup_approx(X + four_q - Y, c.last_w, c.last_ws, q), two_q), q);
  }
  __device__ __forceinline__ void inv_pass_end(V&) const {}
  __device__ __forceinline__ uint64_t fwd_store(V x) const { return csub(csub(csub_n(x, four_q, n4q()), two_q), q); }
  __device__ __forceinline__ uint64_t inv_store(V x) const { return x; }
  __device__ __forceinline__ uint64_t raw(V x) const { return x; }
  __device__ __forceinline__ V unraw(uint64_t x) const { return x; }
};

// q = 2^60 - c (pm_prime). Forward values: below 4q as loaded, below 16q
// between passes; a butterfly takes any 64-bit Y, and adds T < 2.5q to X or 3q
// - T: with X folded (below 1.1q) in the first stage of a pass of at most four,
// or below 4q at the first pass, no value reaches 16q. Inverse values: below
// 8q between passes.
struct PmArith {
  using V = uint64_t;
  using Tw = PmTw;
  uint64_t q, q3, q8;
  uint32_t c, c2;
  __device__ PmArith(const LimbConst& l) : q(l.q), q3(3 * l.q), q8(8 * l.q), c(l.pm_c), c2(2 * l.pm_c) {}
  __device__ __forceinline__ V load(uint64_t x) const { return x; }
  __device__ __forceinline__ void fwd(V& a, V& b, const Tw& t, bool fold) const {
    const uint64_t X = fold ? pm_fold(a, c) : a;
    const uint64_t T = pm_mul_fixed(b, t, c2);
    a = X + T;
    b = X + q3 - T;
  }
  // small: Y < 3q, else Y < 8q; fold: the sum could pass 8q
  __device__ __forceinline__ void inv(V& a, V& b, const Tw& t, bool small, bool fold) const {
    const uint64_t X = a, Y = b;
    a = fold ? pm_fold(X + Y, c) : X + Y;
    b = pm_mul_fixed(X + (small ? q3 : q8) - Y, t, c2);
  }
  __device__ __forceinline__ void inv_last(V& a, V& b, const LimbConst& l) const {
    const uint64_t X = a, Y = b;
    a = pm_canon(pm_mul_fixed(X + Y, l.pm_n_inv, c2), q, c);
    b = pm_canon(pm_mul_fixed(X + q8 - Y, l.pm_last, c2), q, c);
  }
  __device__ __forceinline__ void inv_pass_end(V&) const {}
  __device__ __forceinline__ uint64_t fwd_store(V x) const { return pm_canon(x, q, c); }
  __device__ __forceinline__ uint64_t inv_store(V x) const { return x; }
  __device__ __forceinline__ uint64_t raw(V x) const { return x; }
  __device__ __forceinline__ V unraw(uint64_t x) const { return x; }
};

// Where a pm inverse pass over the register bits [RB0, RB0 + NS) of 16 values
// folds its sums: every value enters below 8q; a product leaves below 2.5q, a
// folded sum below 1.25q, and a sum of two bounds that passes 8q is folded.
// Bounds in quarters of q.
template <int RB0, int NS>
struct InvPlan {
  bool small[NS][16] = {}, fold[NS][16] = {};
  constexpr InvPlan() {
    int bound[16] = {};
    for (int k = 0; k < 16; ++k) bound[k] = 32;
    for (int s = 0; s < NS; ++s)
      for (int k = 0; k < 16; ++k) {
        const int m = 1 << (RB0 + s);
        if (k & m) continue;
        const int sum = bound[k] + bound[k | m];
        small[s][k] = bound[k | m] <= 12;
        fold[s][k] = sum > 32;
        bound[k] = sum > 32 ? 5 : sum;
        bound[k | m] = 10;
      }
  }
};

struct Fp64Arith {
  using V = double;
  using Tw = Fp64Tw;
  double q, qinv;
  __device__ Fp64Arith(const LimbConst& c) : q(c.qd), qinv(c.qinv) {}
  __device__ __forceinline__ V load(uint64_t x) const { return u64_to_f64(x); }
  // values grow by at most 0.51 q per stage; no reduction needed inside the transform
  __device__ __forceinline__ void fwd(V& a, V& b, const Tw& t, bool) const {
    double X = a;
    double T = mulmod_f64(b, t.w, t.wq, q);
    a = X + T;
    b = X - T;
  }
  // the sum doubles per stage: reduced at the end of every register pass
  __device__ __forceinline__ void inv(V& a, V& b, const Tw& t, bool, bool) const {
    double X = a, Y = b;
    a = X + Y;
    b = mulmod_f64(X - Y, t.w, t.wq, q);
  }
  __device__ __forceinline__ void inv_last(V& a, V& b, const LimbConst& c) const {
    double X = a, Y = b;
    double r0 = mulmod_f64(X + Y, c.n_inv_d, c.n_inv_dq, q);
    double r1 = mulmod_f64(X - Y, c.last_wd, c.last_wdq, q);
    a = r0 < 0.0 ? r0 + q : r0;
    b = r1 < 0.0 ? r1 + q : r1;
  }
  __device__ __forceinline__ void inv_pass_end(V& x) const { x = reduce_f64_signed(x, q, qinv); }
  __device__ __forceinline__ uint64_t fwd_store(V x) const { return f64_to_u64(reduce_f64(x, q, qinv)); }
  __device__ __forceinline__ uint64_t inv_store(V x) const { return f64_to_u64(x); }
  __device__ __forceinline__ uint64_t raw(V x) const { return __builtin_bit_cast(uint64_t, x); }
  __device__ __forceinline__ V unraw(uint64_t x) const { return __builtin_bit_cast(double, x); }
};

// f.template operator()<A>() with the arithmetic of limb lc (uniform over the
// workgroup): Fp64Arith below 2^41, else the chain's BIG (PmArith or IntArith).
// APART: nothing that both begin or end with is merged (the compiler hoists and
// sinks it, and holds its registers through either).
template <class BIG, bool APART = false, class F>
__device__ __forceinline__ void with_arith(const LimbConst& lc, F&& f) {
  if (lc.kind == LIMB_FP64) {
    if constexpr (APART) asm volatile("; fp64 limb");
    f.template operator()<Fp64Arith>();
    if constexpr (APART) asm volatile("; fp64 limb, end");
  } else {
    if constexpr (APART) asm volatile("; limb above 2^41");
    f.template operator()<BIG>();
    if constexpr (APART) asm volatile("; limb above 2^41, end");
  }
}

// a times a prepared operand b (launch_to_montgomery) mod q: below 2q, or on
// pm limbs (a < 2^62, b unchanged) below 4q.
template <class A>
__device__ __forceinline__ uint64_t fixed_mul(uint64_t a, uint64_t b, const BarrettConst& bc) {
  if constexpr (std::is_same_v<A, PmArith>)
    return pm_mul(a, b, (uint32_t)bc.pm_c);
  else
    return mont_mul(a, b, bc);
}

// c0 + c1 s with s prepared: below 3q, or on pm limbs below 1.1q (an operand
// of pm_mul again).
template <class A>
__device__ __forceinline__ uint64_t key_dot(uint64_t c0, uint64_t c1, uint64_t s, const BarrettConst& bc) {
  const uint64_t d = c0 + fixed_mul<A>(c1, s, bc);
  if constexpr (std::is_same_v<A, PmArith>)
    return pm_fold(d, (uint32_t)bc.pm_c);
  else
    return d;
}

// d p - y s for a forward transform's output y (its arithmetic's
// representation) and prepared p and s, in the inverse transform's input range:
// products below 2q leave it in (0, 4q), below 4q (pm limbs) in (0, 8q); the
// FP64 inverse gets it canonical.
template <class A>
__device__ __forceinline__ uint64_t prepared_difference(const A& ar, uint64_t d, uint64_t p, typename A::V y, uint64_t s,
                                                        const BarrettConst& bc) {
  const uint64_t u = fixed_mul<A>(d, p, bc);
  if constexpr (std::is_same_v<A, PmArith>) return u + 4 * ar.q - fixed_mul<A>(pm_fold(y, ar.c), s, bc);
  const uint64_t e = u + 2 * bc.q - fixed_mul<A>(ar.fwd_store(y), s, bc);
  return std::is_same_v<A, Fp64Arith> ? csub(csub(e, 2 * bc.q), bc.q) : e;
}

// (m - r) q_last^{-1} mod q, canonical, from the canonical coefficient m and
// the last limb's coefficient r: reduced mod q, or on pm limbs as it is (below
// 2^61 < 3q).
template <class A>
__device__ __forceinline__ uint64_t rescaled_coefficient(uint64_t m, uint64_t r, const RescaleConst& rc,
                                                         const LimbConst& lc) {
  if constexpr (std::is_same_v<A, PmArith>)
    return pm_canon(pm_mul_fixed(m + 3 * lc.q - r, rc.pm_inv, 2 * lc.pm_c), lc.q, lc.pm_c);
  else
    return csub(shoup_lazy(submod(m, r, lc.q), rc.inv, rc.inv_s, lc.q), lc.q);
}

// The operation fused into the coefficient load (NttLoad), fixed at compile
// time so that each kernel carries only its own operation; `i` indexes the
// limb-polynomial, so src, aux and key are read at the same position.
template <uint32_t LD>
struct LoadOp {
  const uint64_t* aux;
  const uint64_t* key;  // secret-key limb-poly (DOT)
  BarrettConst bc;
  RescaleConst rc;
  uint32_t sub;         // ENC variant (uniform over the job)
  double qd, qinv;      // q and 1/q as doubles (ENC)
  // Values a load leaves for the transform: canonical on the Int and Fp64
  // limbs (MULM below 2q, DOTM below 3q), below 4q forward and 8q inverse on
  // pm limbs.
  // signed_residue_dev with |e| in [q, 2^52) reduced by one exact FP64 step:
  // quot = rint(|e| / q) is within one of the true quotient, and the remainder
  // fma(-quot, q, |e|) is an exact integer in (-q, q)
  __device__ __forceinline__ uint64_t enc_residue(int64_t e) const {
    const uint64_t a = e >= 0 ? (uint64_t)e : (uint64_t)0 - (uint64_t)e;
    uint64_t r = a;
    if (a >= bc.q) {
      if (a < (1ULL << 52)) {
        const double ad = u64_to_f64(a);
        double t = __fma_rn(-__builtin_rint(ad * qinv), qd, ad);
        t = t < 0.0 ? t + qd : t;
        r = f64_to_u64(t >= qd ? t - qd : t);
      } else {
        r = mulmod_barrett(a, 1, bc);
      }
    }
    return e >= 0 ? r : bc.q - r;
  }
  // MULM and ENC in two steps, so that a pass issues all 16 of a thread's
  // operand loads before any arithmetic (the per-element branches of the
  // residue forms would otherwise hold each load until the previous
  // element's result): fetch16 reads the operands of positions idx(0..15),
  // finish forms one position's value. MULM reads (ct, pt); ENC, by the
  // job's variant, the ternary byte (2), m or e1 (1), or m and e0 (0).
  static constexpr uint32_t kind = LD;
  struct Raw {
    uint64_t x, a;
  };
  __device__ __forceinline__ Raw fetch(const uint64_t* src, uint32_t i) const {
    static_assert(LD == NTT_LOAD_MULM || LD == NTT_LOAD_ENC, "two-step loads are for MULM and ENC");
    if constexpr (LD == NTT_LOAD_ENC) {
      if (sub == 2) return Raw{gld(reinterpret_cast<const uint8_t*>(src))[i], 0};
      return Raw{gld(src)[i], sub == 0 ? gld(aux)[i] : 0};
    } else {
      return Raw{gld(src)[i], gld(aux)[i]};
    }
  }
  // the variant test outside the element loop, so the 16 requests issue together
  template <class Idx>
  __device__ __forceinline__ void fetch16(const uint64_t* src, const Idx& idx, Raw (&r)[16]) const {
    static_assert(LD == NTT_LOAD_MULM || LD == NTT_LOAD_ENC, "two-step loads are for MULM and ENC");
    const GPtr<uint64_t> s = gld(src);
    if constexpr (LD == NTT_LOAD_ENC) {
      if (sub == 2) {
        const GPtr<uint8_t> u = gld(reinterpret_cast<const uint8_t*>(src));
#pragma unroll
        for (int k = 0; k < 16; ++k) r[k] = Raw{u[idx(k)], 0};
      } else if (sub == 0) {
        const GPtr<uint64_t> e = gld(aux);
#pragma unroll
        for (int k = 0; k < 16; ++k) r[k] = Raw{s[idx(k)], e[idx(k)]};
      } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) r[k] = Raw{s[idx(k)], 0};
      }
    } else {
      const GPtr<uint64_t> a = gld(aux);
#pragma unroll
      for (int k = 0; k < 16; ++k) r[k] = Raw{s[idx(k)], a[idx(k)]};
    }
  }
  template <class A>
  __device__ __forceinline__ uint64_t finish(const Raw& r) const {
    if constexpr (LD == NTT_LOAD_ENC) {
      if (sub == 2) return r.x == 0 ? bc.q - 1 : (r.x == 1 ? 0 : 1);
      if constexpr (std::is_same_v<A, PmArith>) {
        // one fold per signed operand, its 8c taken out again: below 3.1q
        const uint32_t c = (uint32_t)bc.pm_c;
        const uint64_t v = pm_fold_signed((int64_t)r.x, c);
        return sub == 0 ? v + pm_fold_signed((int64_t)r.a, c) + (bc.q - 16 * bc.pm_c) : v + (bc.q - 8 * bc.pm_c);
      }
      const uint64_t v = enc_residue((int64_t)r.x);
      return sub == 0 ? csub(v + enc_residue((int64_t)r.a), bc.q) : v;
    } else {
      return fixed_mul<A>(r.x, r.a, bc);
    }
  }
  template <class A>
  __device__ __forceinline__ uint64_t at(const uint64_t* src, uint32_t i) const {
    constexpr bool PM = std::is_same_v<A, PmArith>;
    if constexpr (LD == NTT_LOAD_ENC || LD == NTT_LOAD_MULM) return finish<A>(fetch(src, i));
    const uint64_t x = gld(src)[i];
    if constexpr (LD == NTT_LOAD_DOTM) return x + fixed_mul<A>(gld(aux)[i], gld(key)[i], bc);
    if constexpr (LD == NTT_LOAD_MUL) {
      if constexpr (PM)
        return pm_mul(x, gld(aux)[i], (uint32_t)bc.pm_c);
      else
        return mulmod_barrett(x, gld(aux)[i], bc);
    }
    if constexpr (LD == NTT_LOAD_REDUCE) return PM || x < rc.q ? x : mulmod_barrett(x, 1, rc.b);  // pm: x < 2^61 < 3q
    if constexpr (LD == NTT_LOAD_DOT) {
      if constexpr (PM)
        return x + pm_mul(gld(aux)[i], gld(key)[i], (uint32_t)bc.pm_c);
      else
        return addmod(x, mulmod_barrett(gld(aux)[i], gld(key)[i], bc), bc.q);
    }
    return x;
  }
};

// The operation fused into a forward transform's final store (NttStore), or,
// for SEGSUM, the inverse transform's segment-sum epilogue's operands.
template <uint32_t ST>
struct StoreOp {
  static constexpr uint32_t kind = ST;
  const uint64_t* aux;
  const uint64_t* aux2;
  BarrettConst bc;
  RescaleConst rc;
  const double* segw;  // SEGSUM
  double* seg;
  double scale;
  uint32_t cols;
  // Operands the store reads at position i (ct x pt factors, or the value the
  // rescale subtracts from); loaded apart from the arithmetic so that a pass
  // can issue these loads early and hide their latency behind its butterflies.
  static constexpr int NAUX = ST == NTT_STORE_MUL_RESCALE ? 2 : ST == NTT_STORE_RESCALE ? 1 : 0;
  // Store of transform output x at position i of dst (MONT: its Montgomery
  // form, and the plain residue to aux when aux is set).
  template <class A>
  __device__ __forceinline__ void store(const A& ar, typename A::V x, GMut<uint64_t> dst, uint32_t i,
                                        uint64_t cp) const {
    if constexpr (ST == NTT_STORE_MONT) {
      const uint64_t y = ar.fwd_store(x);
      if constexpr (std::is_same_v<A, PmArith>)
        dst[i] = y;
      else
        dst[i] = csub(shoup_lazy(y, bc.r64, bc.r64_s, bc.q), bc.q);  // y 2^64 mod q
      if (aux) gst(const_cast<uint64_t*>(aux))[i] = y;
    } else {
      dst[i] = apply_prep(ar, x, cp);
    }
  }
  struct Aux {
    uint64_t a, b;
  };
  __device__ __forceinline__ Aux load_aux(uint32_t i) const {
    Aux v{0, 0};
    if constexpr (NAUX >= 1) v.a = gld(aux)[i];
    if constexpr (NAUX >= 2) v.b = gld(aux2)[i];
    return v;
  }
  // The value the rescale subtracts from (ct x pt product, or the single
  // operand), reduced modulo q, from the operands v: a double's bit pattern
  // on limbs below 2^41 (Fp64Arith), else the residue (below 4q on pm limbs).
  template <class A>
  __device__ __forceinline__ uint64_t prep(const A&, const Aux& v) const {
    if constexpr (NAUX == 0) {
      return 0;
    } else if constexpr (std::is_same_v<A, Fp64Arith>) {
      double c;
      if constexpr (ST == NTT_STORE_MUL_RESCALE)
        c = mulmod_f64_any(u64_to_f64(v.a), u64_to_f64(v.b), rc.qd, rc.qinv);
      else
        c = u64_to_f64(v.a);
      return __builtin_bit_cast(uint64_t, c);
    } else {
      if constexpr (ST != NTT_STORE_MUL_RESCALE)
        return v.a;
      else if constexpr (std::is_same_v<A, PmArith>)
        return pm_mul(v.a, v.b, (uint32_t)bc.pm_c);
      else
        return mulmod_barrett(v.a, v.b, bc);
    }
  }
  // The stored word for transform output x (the arithmetic's representation)
  // with the prepared value c of its position (prep). Limbs below 2^41
  // (Fp64Arith) do the rescale in doubles: exact products without
  // precomputed companions instead of 64-bit Barrett.
  template <class A>
  __device__ __forceinline__ uint64_t apply_prep(const A& ar, typename A::V x, uint64_t cp) const {
    if constexpr (std::is_same_v<A, Fp64Arith> && NAUX > 0) {
      // (c - x) * inv with the output as it is: |x| < 9 q + 2^32 (the input,
      // reduce_u64_f64, and at most 15 stages of 0.51 q), so |c - x| < 2^46
      const double c = __builtin_bit_cast(double, cp);
      const double r = mulmod_f64(c - x, rc.inv_d, rc.inv_dq, rc.qd);
      return f64_to_u64(r < 0.0 ? r + rc.qd : r);
    } else if constexpr (std::is_same_v<A, PmArith> && NAUX > 0) {
      // cp < 4q, the folded output below 2q
      return pm_canon(pm_mul_fixed(cp + 2 * ar.q - pm_fold(x, ar.c), rc.pm_inv, ar.c2), ar.q, ar.c);
    } else {
      const uint64_t y = ar.fwd_store(x);
      if constexpr (NAUX == 0)
        return y;
      else
        return csub(shoup_lazy(submod(cp, y, rc.q), rc.inv, rc.inv_s, rc.q), rc.q);
    }
  }
};

// Load and store operations of job `jb` in launch `a` for limb `limb`.
template <uint32_t LD, uint32_t ST>
__device__ __forceinline__ void job_ops(const NttArgs& a, const NttJob& jb, uint32_t limb, uint32_t n,
                                        LoadOp<LD>& op, StoreOp<ST>& so) {
  op.aux = jb.aux;
  if constexpr (LD == NTT_LOAD_MUL || LD == NTT_LOAD_DOT || LD == NTT_LOAD_ENC || LD == NTT_LOAD_MULM ||
                LD == NTT_LOAD_DOTM)
    op.bc = a.bc[limb];
  if constexpr (LD == NTT_LOAD_ENC) {
    op.sub = jb.sub;
    op.qd = a.lc[limb].qd;
    op.qinv = a.lc[limb].qinv;
  }
  if constexpr (LD == NTT_LOAD_DOT || LD == NTT_LOAD_DOTM) op.key = a.key + (uint64_t)limb * n;
  if constexpr (LD == NTT_LOAD_REDUCE) op.rc = a.rc[limb];
  so.aux = jb.aux;
  so.aux2 = jb.aux2;
  if constexpr (ST == NTT_STORE_RESCALE || ST == NTT_STORE_MUL_RESCALE) so.rc = a.rc[limb];
  if constexpr (ST == NTT_STORE_MUL_RESCALE || ST == NTT_STORE_MONT) so.bc = a.bc[limb];
  if constexpr (ST == NTT_STORE_SEGSUM) {
    so.segw = a.segw;
    so.seg = reinterpret_cast<double*>(jb.dst);
    so.scale = jb.scale;
    so.cols = a.cols;
  }
}

// Calls f.template operator()<LD, ST>() for the (load, store) pair of a launch.
// Only the pairs the engine issues are instantiated: forward (NONE | ENC,
// NONE), (REDUCE, RESCALE), (REDUCE, MUL_RESCALE), (NONE, MONT); inverse
// (NONE | MUL | MULM | DOT | DOTM, NONE), (DOT | DOTM, SEGSUM).
template <bool INV, class F>
__host__ hipError_t with_ops(uint32_t load, uint32_t store, F&& f) {
  if constexpr (!INV) {
    if (load == NTT_LOAD_NONE && store == NTT_STORE_NONE) return f.template operator()<NTT_LOAD_NONE, NTT_STORE_NONE>();
    if (load == NTT_LOAD_ENC && store == NTT_STORE_NONE) return f.template operator()<NTT_LOAD_ENC, NTT_STORE_NONE>();
    if (load == NTT_LOAD_REDUCE && store == NTT_STORE_RESCALE)
      return f.template operator()<NTT_LOAD_REDUCE, NTT_STORE_RESCALE>();
    if (load == NTT_LOAD_REDUCE && store == NTT_STORE_MUL_RESCALE)
      return f.template operator()<NTT_LOAD_REDUCE, NTT_STORE_MUL_RESCALE>();
    if (load == NTT_LOAD_NONE && store == NTT_STORE_MONT) return f.template operator()<NTT_LOAD_NONE, NTT_STORE_MONT>();
    return hipErrorInvalidValue;
  } else {
    if (load == NTT_LOAD_DOT && store == NTT_STORE_SEGSUM)
      return f.template operator()<NTT_LOAD_DOT, NTT_STORE_SEGSUM>();
    if (load == NTT_LOAD_DOTM && store == NTT_STORE_SEGSUM)
      return f.template operator()<NTT_LOAD_DOTM, NTT_STORE_SEGSUM>();
    if (store != NTT_STORE_NONE) return hipErrorInvalidValue;
    if (load == NTT_LOAD_NONE) return f.template operator()<NTT_LOAD_NONE, NTT_STORE_NONE>();
    if (load == NTT_LOAD_MUL) return f.template operator()<NTT_LOAD_MUL, NTT_STORE_NONE>();
    if (load == NTT_LOAD_MULM) return f.template operator()<NTT_LOAD_MULM, NTT_STORE_NONE>();
    if (load == NTT_LOAD_DOT) return f.template operator()<NTT_LOAD_DOT, NTT_STORE_NONE>();
    if (load == NTT_LOAD_DOTM) return f.template operator()<NTT_LOAD_DOTM, NTT_STORE_NONE>();
    return hipErrorInvalidValue;
  }
}

}  // namespace th
