// Device-side definitions shared by the HIP kernels of the CKKS engine.
//
// Residues live in HBM as canonical u64 values in [0, q), limb-major:
// a limb-polynomial is N consecutive u64, a ciphertext is [c0 | c1] with each
// component L limb-polynomials back to back (the reference's RnsPoly layout,
// tensafe-he-core/src/rns.rs:199-206, made contiguous).
//
// Three exact modular-multiply paths are used, chosen per prime (LimbKind):
//  * "int":  64-bit Shoup multiply with a precomputed floor(w*2^64/q) and
//            Harvey-style lazy reduction; any q < 2^61.
//  * "fp64": for q < 2^41 the product w*x is split exactly into hi + lo with
//            one FMA and the quotient comes from x*(w/q) rounded to nearest;
//            the remainder is exact (all intermediate integers < 2^53). Six
//            full-rate FP64 instructions per multiply.
//  * "pm":   for q = 2^60 - c with a small c (the 60-bit primes of every
//            default chain) 2^60 = c mod q, so a product is folded at bit 60
//            instead of divided: no quotient is formed. 12 instructions per
//            product by a fixed operand against the Shoup product's 14 and,
//            since one fold takes any 64-bit value below q + 16 c, a forward
//            butterfly of 16 instructions (one fold of half the values every
//            four stages) against 22 with a conditional subtraction each.
// All produce the unique canonical residue, so results are bit-identical to
// the reference's u128 Barrett multiply (tensafe-he-core/src/rns.rs:45-95).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace th {

// Largest prime that takes the fp64 multiply path.
constexpr uint64_t FP64_PRIME_LIMIT = 1ULL << 41;

// A prime q takes the pm path when 2^60 - 2^26 < q < 2^60.
constexpr uint64_t PM_MAX_C = 1ULL << 26;
constexpr bool pm_prime(uint64_t q) { return q < (1ULL << 60) && q > (1ULL << 60) - PM_MAX_C; }
enum LimbKind : uint32_t { LIMB_INT = 0, LIMB_FP64 = 1, LIMB_PM = 2 };

// A fixed operand w < q of a pm product in 30-bit halves, w = wl + wh 2^30,
// beside v = w 2^32 mod q likewise: x w = x0 w + x1 v (mod q) for the 32-bit
// halves of x, and no sum of two partial products passes 2^63.
struct PmTw {
  uint32_t wl, wh, vl, vh;
};
struct ShoupTw {
  uint64_t w, ws;  // twiddle and floor(w * 2^64 / q)
};
struct Fp64Tw {
  double w, wq;  // twiddle and w / q (correctly rounded)
};

// Per-limb constants; one array per context in device memory.
struct LimbConst {
  uint64_t q, two_q;
  uint64_t n_inv, n_inv_s;    // N^{-1} and its Shoup companion
  uint64_t last_w, last_ws;   // inv_tw[1] * N^{-1}: last inverse stage with the scaling folded in
  double qd, qinv;            // q and 1/q as doubles (fp64 path)
  double n_inv_d, n_inv_dq;
  double last_wd, last_wdq;
  PmTw pm_n_inv, pm_last;     // n_inv and last_w for the pm path
  const void* fwd;            // N twiddle pairs (ShoupTw, Fp64Tw or PmTw), fwd[brv(i)] = psi^i
  const void* inv;            // N twiddle pairs, inv[brv(i)] = psi^-i
  const void* fwd_row;        // fwd and inv entries of the split row passes' lane-bit stages
  const void* inv_row;        //   in the order their lanes read them (row_table_index)
  uint32_t kind;              // LimbKind
  uint32_t pm_c;              // 2^60 - q (pm path)
};

// A context's limb constants in device memory, and whether its chain takes the
// pm path: every prime is a pm prime or below 2^41. Chains that mix in other
// large primes take the int path for all of them, so each transform kernel
// carries two arithmetics, fp64 and one of int and pm.
struct LimbTable {
  LimbConst* p = nullptr;
  uint32_t pm = 0;
  __device__ __forceinline__ const LimbConst& operator[](uint32_t l) const { return p[l]; }
};

// ---------------------------------------------------------------- int path
__device__ __forceinline__ uint64_t shoup_lazy(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
  // x * w mod q in [0, 2q) for any x < 2^64 (w < q).
  uint64_t qh = __umul64hi(x, ws);
  return x * w - qh * q;
}

__device__ __forceinline__ uint64_t csub(uint64_t x, uint64_t m) { return x >= m ? x - m : x; }

// The same with nm = 2^64 - m supplied: x + nm is one 64-bit add (no borrow
// chain through VCC), and the compare selects between x and the sum.
__device__ __forceinline__ uint64_t csub_n(uint64_t x, uint64_t m, uint64_t nm) {
  const uint64_t t = x + nm;
  return x >= m ? t : x;
}

// v unchanged, but hidden from the optimiser (an empty asm that claims to
// modify it), so that 2^64 - m stays an addend instead of being folded back
// into a subtraction of m.
__device__ __forceinline__ uint64_t opaque_u64(uint64_t v) {
  asm("" : "+v"(v));
  return v;
}

// Pointers known to address global memory (address space 1). Pointers read
// from job descriptors or constant tables are generic to the compiler, and
// generic (flat) loads and stores also count against the LDS wait counter,
// which serialises them with every LDS exchange; accesses through these
// pointers are global_* instructions instead.
template <class T>
using GPtr = const __attribute__((address_space(1))) T*;
template <class T>
using GMut = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ GPtr<T> gld(const T* p) {
  return (GPtr<T>)p;
}
template <class T>
__device__ __forceinline__ GMut<T> gst(T* p) {
  return (GMut<T>)p;
}
// Element i of a global array of 16-byte records (twiddle pairs), loaded as one
// 16-byte vector.
template <class T>
__device__ __forceinline__ T ld16(GPtr<T> p, uint32_t i) {
  static_assert(sizeof(T) == 16, "16-byte records only");
  using V = uint64_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(T, ((GPtr<V>)p)[i]);
}
// The same through the constant address space, for an index that is the same
// on every lane of the wavefront: a scalar load, which leaves the CU's
// vector-memory path to the per-lane accesses (only for tables that no kernel
// writes while it runs).
template <class T>
__device__ __forceinline__ T ld16_uniform(GPtr<T> p, uint32_t i) {
  static_assert(sizeof(T) == 16, "16-byte records only");
  using V = uint64_t __attribute__((ext_vector_type(2)));
  using CPtr = const __attribute__((address_space(4))) V*;
  return __builtin_bit_cast(T, ((CPtr)(const void*)p)[__builtin_amdgcn_readfirstlane(i)]);
}

// floor(x * s / 2^64) - e with e in {0, 1, 2}: x1*s1 + hi(x1*s0) + hi(x0*s1)
// for 32-bit halves; the low halves of the two cross products and hi(x0*s0)
// are dropped, each below 2^32, so at most 2 is lost after the shift. The sum
// stays below 2^64. The last term goes in as a 32-bit add with carry (two
// 32-bit instructions): left to the compiler it becomes a zero-extending move
// and a 64-bit add.
__device__ __forceinline__ uint64_t mulhi_approx(uint64_t x, uint64_t s) {
  const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32), s0 = (uint32_t)s, s1 = (uint32_t)(s >> 32);
  const uint64_t r = (uint64_t)x1 * s1 + __umulhi(x1, s0);
  uint32_t rl = (uint32_t)r, rh = (uint32_t)(r >> 32);
  asm("v_add_co_u32 %0, vcc, %0, %2\n\tv_addc_co_u32 %1, vcc, %1, 0, vcc" : "+v"(rl), "+v"(rh) : "v"(__umulhi(x0, s1))
      : "vcc");
  return ((uint64_t)rh << 32) | rl;
}

// v unchanged, hidden from the optimiser (see opaque_u64).
__device__ __forceinline__ uint32_t opaque_u32(uint32_t v) {
  asm("" : "+v"(v));
  return v;
}

// x * w mod q in [0, 4q) for any 64-bit x (w < q, ws = floor(w * 2^64 / q)):
// the exact Shoup remainder is below 2q and the quotient estimate is at most
// 2 short.
// The remainder is formed as x*w + qhat*(2^64 - q) mod 2^64 from 32-bit
// partial products, so that the second low product accumulates onto the first
// (one multiply-add) instead of being subtracted as a separate 64-bit word.
__device__ __forceinline__ uint64_t shoup_approx(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
  const uint64_t qh = mulhi_approx(x, ws);
  const uint64_t nq = 0 - q;
  const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32), w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32);
  const uint32_t h0 = (uint32_t)qh, h1 = (uint32_t)(qh >> 32), n0 = (uint32_t)nq, n1 = (uint32_t)(nq >> 32);
  const uint64_t lo = (uint64_t)x0 * w0 + (uint64_t)h0 * n0;
  // the high word as one 32-bit sum (the cross products pair up as multiply-
  // adds); kept opaque so that the compiler does not turn the word assembly
  // back into a 64-bit add of the shifted cross terms
  const uint32_t hi = opaque_u32((uint32_t)(lo >> 32) + (x0 * w1 + x1 * w0) + (h0 * n1 + h1 * n0));
  return ((uint64_t)hi << 32) | (uint32_t)lo;
}

// Exact a*b mod q for a, b < q < 2^63 (operands without a precomputed
// companion): 128-bit product, quotient from the high word scaled by a
// per-prime reciprocal, then at most two corrections.
struct BarrettConst {
  uint64_t q;
  uint64_t r_hi, r_lo;  // floor((2^128 - 1) / q) as two words
  uint64_t mq;          // -q^{-1} mod 2^64 (Montgomery products)
  uint64_t r64;         // 2^64 mod q (into Montgomery form)
  uint64_t r64_s;       // floor(r64 2^64 / q): its Shoup companion
  uint64_t pm_c;        // 2^60 - q on the pm path, else 0
  double qd, qinv;      // q and 1/q as doubles below 2^41, else 0
};

__device__ __forceinline__ uint64_t mulmod_barrett(uint64_t a, uint64_t b, const BarrettConst& m) {
  uint64_t lo = a * b;
  uint64_t hi = __umul64hi(a, b);
  // quotient estimate = floor((hi*2^64 + lo) * (r_hi*2^64 + r_lo) / 2^128), lo*r_lo term dropped
  uint64_t t1_lo = lo * m.r_hi, t1_hi = __umul64hi(lo, m.r_hi);
  uint64_t t2_lo = hi * m.r_lo, t2_hi = __umul64hi(hi, m.r_lo);
  uint64_t mid = t1_lo + t2_lo;
  uint64_t carry = mid < t1_lo ? 1 : 0;
  uint64_t quot = hi * m.r_hi + t1_hi + t2_hi + carry;
  uint64_t r = lo - quot * m.q;
  r = csub(r, m.q);
  r = csub(r, m.q);
  return r;
}

__device__ __forceinline__ uint64_t addmod(uint64_t a, uint64_t b, uint64_t q) { return csub(a + b, q); }

// Montgomery product a * b * 2^-64 mod q in [0, 2q) for any 64-bit a and
// b < q: with T = a b and m = T mod 2^64 * (-q^{-1}) mod 2^64, T + m q is a
// multiple of 2^64, its low words cancel (a carry exactly when T mod 2^64 is
// nonzero), and (T + m q) / 2^64 < 2q. With b = w 2^64 mod q (w in Montgomery
// form) this is a * w mod q, in about half the multiplies of a Barrett product.
__device__ __forceinline__ uint64_t mont_mul(uint64_t a, uint64_t b, const BarrettConst& m) {
  const uint64_t t_lo = a * b, t_hi = __umul64hi(a, b);
  const uint64_t k = t_lo * m.mq;
  return t_hi + __umul64hi(k, m.q) + (t_lo != 0 ? 1 : 0);
}

// e >= 0 ? e mod q : q - (|e| mod q) (ciphertext.rs:132-136, :275-287; encoding.rs:198-202)
__device__ __forceinline__ uint64_t signed_residue_dev(int64_t e, const BarrettConst& m) {
  const uint64_t a = e >= 0 ? (uint64_t)e : (uint64_t)0 - (uint64_t)e;
  const uint64_t r = a < m.q ? a : mulmod_barrett(a, 1, m);
  return e >= 0 ? r : m.q - r;
}

__device__ __forceinline__ uint64_t submod(uint64_t a, uint64_t b, uint64_t q) {
  return a >= b ? a - b : a + q - b;
}

// ---------------------------------------------------------------- pm path
// q = 2^60 - c, 0 < c < 2^26.
//
// x mod q, below q + 16 c, for any 64-bit x: the bits from 60 on fold to
// multiples of c (three instructions).
__device__ __forceinline__ uint64_t pm_fold(uint64_t x, uint32_t c) {
  const uint32_t h = (uint32_t)(x >> 32);
  return (uint64_t)(h >> 28) * c + (((uint64_t)(h & 0x0fffffffu) << 32) | (uint32_t)x);
}
// x mod q, canonical, for any 64-bit x.
__device__ __forceinline__ uint64_t pm_canon(uint64_t x, uint64_t q, uint32_t c) {
  return csub_n(pm_fold(x, c), q, opaque_u64(0 - q));
}
// x w mod q in [0, 2.5 q) for any 64-bit x. With ab = x0 wl + x1 vl and
// cd = x0 wh + x1 vh (each at most 2^63 - 2^33 - 2^31 + 2: no overflow) the
// product is ab + cd 2^30; its bits from 61 on, cd >> 31 (at most 2^32 - 5)
// plus the at most 4 from the lower part's sum, are one 32-bit word h, and
// h 2^61 = 2 h c. The result is below 2^61 + 2^32 2c <= 2^61 + 2^59.
__device__ __forceinline__ uint64_t pm_mul_fixed(uint64_t x, const PmTw& t, uint32_t c2) {
  const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32);
  const uint64_t ab = (uint64_t)x1 * t.vl + (uint64_t)x0 * t.wl;
  const uint64_t cd = (uint64_t)x1 * t.vh + (uint64_t)x0 * t.wh;
  const uint32_t top = __builtin_amdgcn_alignbit((uint32_t)(cd >> 32), (uint32_t)cd, 31);
  const uint64_t d = ((uint64_t)((uint32_t)cd & 0x7fffffffu) << 30) + ab;
  const uint32_t dh = (uint32_t)(d >> 32);
  const uint32_t h = top + (dh >> 29);
  return (uint64_t)h * c2 + (((uint64_t)(dh & 0x1fffffffu) << 32) | (uint32_t)d);
}
// a b mod q in [0, 4q) for a < 2^62, b < 2^60, neither with a companion: from
// 30-bit halves a b = p11 2^60 + mid 2^30 + p00, and with mid = mh 2^30 + ml
//   a b = (p11 + mh) c + ml 2^30 + p00  (mod q).
// (p11 + mh) c has up to 88 bits: e0 c below, y = e1 c (< 2^57) times 2^32
// above, whose bits from 28 on fold once more. Every term is below 2^60 + 2^58.
__device__ __forceinline__ uint64_t pm_mul(uint64_t a, uint64_t b, uint32_t c) {
  constexpr uint32_t M30 = (1u << 30) - 1, M28 = (1u << 28) - 1;
  const uint32_t a0 = (uint32_t)a & M30, b0 = (uint32_t)b & M30;
  const uint32_t a1 = __builtin_amdgcn_alignbit((uint32_t)(a >> 32), (uint32_t)a, 30);
  const uint32_t b1 = __builtin_amdgcn_alignbit((uint32_t)(b >> 32), (uint32_t)b, 30);
  const uint64_t p00 = (uint64_t)a0 * b0, mid = (uint64_t)a1 * b0 + (uint64_t)a0 * b1;
  const uint64_t e = (uint64_t)a1 * b1 + (mid >> 30);
  const uint32_t ml = (uint32_t)mid & M30;
  const uint64_t r = ((uint64_t)ml << 30) + p00 + (uint64_t)(uint32_t)e * c;
  const uint64_t y = (uint64_t)(uint32_t)(e >> 32) * c;
  const uint32_t yh = __builtin_amdgcn_alignbit((uint32_t)(y >> 32), (uint32_t)y, 28);
  return r + ((uint64_t)((uint32_t)y & M28) << 32) + (uint64_t)yh * c;
}
// A residue of e + 8c, below q + 16 c, for any signed e: e + 2^63 is unsigned,
// and 2^63 = 8c (mod q).
__device__ __forceinline__ uint64_t pm_fold_signed(int64_t e, uint32_t c) {
  return pm_fold((uint64_t)e ^ (1ULL << 63), c);
}

// Operands fixed for many products are kept prepared for the limb's general
// product: Montgomery form, except on the pm path, which takes them as they
// are (launch_to_montgomery). a * prepared(b) mod q, a < 2^62: below 2q from
// the Montgomery product, below 4q from the pm product.
__device__ __forceinline__ uint64_t prepared_mul(uint64_t a, uint64_t b, const BarrettConst& m) {
  return m.pm_c ? pm_mul(a, b, (uint32_t)m.pm_c) : mont_mul(a, b, m);
}

// Rescale constants of one output limb l (ciphertext.rs:497-522).
struct RescaleConst {
  uint64_t q, inv, inv_s;  // q_l, (q_last mod q_l)^{-1} and its Shoup companion
  BarrettConst b;          // remainder of a 64-bit value modulo q_l
  double qd, qinv;         // q_l and 1/q_l as doubles (limbs below 2^41)
  double inv_d, inv_dq;    // inv and inv / q_l as doubles (limbs below 2^41)
  double q32, r32;         // q_l / 2^32 (exact) and 2^32 / q_l (limbs below 2^41)
  PmTw pm_inv;             // inv for the pm path
};

// ---------------------------------------------------------------- fp64 path
// x*w mod q as an exact integer in about (-q/2, q/2); requires |x| < 2^46, w < q < 2^41.
__device__ __forceinline__ double mulmod_f64(double x, double w, double wq, double q) {
  double hi = x * w;
  double lo = __fma_rn(x, w, -hi);
  double quot = __builtin_rint(x * wq);
  double r = __fma_rn(-quot, q, hi);
  return r + lo;
}

// A residue of any c < 2^61 modulo a limb q_l below 2^41, as an exact double
// of magnitude below 0.76 q_l + 2^32 (0.52 q_l + 2^32 from q_l = 2^21 on, 2^32
// being most of it for a small q_l), the forward transforms' input: with c =
// ch 2^32 + cl (ch < 2^29) and quot = rint(ch 2^32 / q_l), ch - quot q_l / 2^32
// is an exact multiple of 2^-32 (one FMA), and times 2^32 plus cl the residue
// (another). Six instructions; through 2^32 mod q_l and corrected into [0,
// q_l) it took 17, a third of the rescale column kernel's instructions on
// these limbs.
__device__ __forceinline__ double reduce_u64_f64(uint64_t c, const RescaleConst& rc) {
  const double ch = (double)(uint32_t)(c >> 32), cl = (double)(uint32_t)c;
  const double quot = __builtin_rint(ch * rc.r32);
  return __fma_rn(__fma_rn(-quot, rc.q32, ch), 0x1p32, cl);
}

// a*b mod q within 0.51 q of zero for integers 0 <= a, b < q < 2^41 held
// exactly in doubles, without a precomputed companion: hi + lo = a*b exactly
// (one FMA), and quot = rint(hi / q) through qinv = 1/q is within 0.5 + 2^-10
// of a*b/q (a*b/q < 2^41, relative error below 2^-51), and a*b - quot*q is
// formed exactly.
__device__ __forceinline__ double mulmod_f64_any(double a, double b, double q, double qinv) {
  const double hi = a * b;
  const double lo = __fma_rn(a, b, -hi);
  const double quot = __builtin_rint(hi * qinv);
  return __fma_rn(-quot, q, hi) + lo;
}

// x mod q into [0, q) for an exact integer |x| < 2^50.
__device__ __forceinline__ double reduce_f64(double x, double q, double qinv) {
  double quot = __builtin_rint(x * qinv);
  double r = __fma_rn(-quot, q, x);
  return r < 0.0 ? r + q : r;
}

// x mod q into about (-q/2, q/2) (no sign fix) for an exact integer |x| < 2^50.
__device__ __forceinline__ double reduce_f64_signed(double x, double q, double qinv) {
  double quot = __builtin_rint(x * qinv);
  return __fma_rn(-quot, q, x);
}

// Between integers 0 <= x < 2^52 and doubles through the bits of 2^52 + x: two
// instructions each way (the general conversions take four and six).
__device__ __forceinline__ double u64_to_f64(uint64_t x) {
  return __builtin_bit_cast(double, x | 0x4330000000000000ULL) - 0x1p52;
}
__device__ __forceinline__ uint64_t f64_to_u64(double x) {
  return __builtin_bit_cast(uint64_t, x + 0x1p52) & 0x000fffffffffffffULL;
}

// a * b mod q, canonical, for canonical operands on any limb: the limb's own
// product (about 16 instructions below 2^41, 27 on pm limbs), Barrett's (about
// 50) on the others.
__device__ __forceinline__ uint64_t mulmod(uint64_t a, uint64_t b, const BarrettConst& m) {
  if (m.qd != 0.0) {
    const double r = mulmod_f64_any(u64_to_f64(a), u64_to_f64(b), m.qd, m.qinv);
    return f64_to_u64(r < 0.0 ? r + m.qd : r);
  }
  if (m.pm_c) return pm_canon(pm_mul(a, b, (uint32_t)m.pm_c), m.q, (uint32_t)m.pm_c);
  return mulmod_barrett(a, b, m);
}

}  // namespace th
