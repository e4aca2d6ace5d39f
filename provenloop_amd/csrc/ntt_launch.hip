// Which transform kernels a batch takes, by its size and its chain's arithmetic
// (LimbTable::pm). Two kernel families. ntt.hip: one workgroup transforms one
// limb-polynomial on chip (N <= 16384). ntt_split.hip: a column pass plus a row
// pass of single-wavefront workgroups (N >= 8192). The whole-polynomial kernel
// moves each coefficient through HBM once but, at N = 16384, fills a CU's LDS,
// so a CU cannot overlap one polynomial's loads with another's arithmetic; the
// split kernels move the data twice but keep many wavefronts per CU. The whole-
// polynomial kernel's time grows in steps of one round of workgroups (one per
// CU) and a round takes a transform's time however few workgroups it holds,
// while the split kernels spread every transform over 16 workgroups. Measured on
// MI355X at N = 16384 (forward, 4-limb chain): 4 transforms 23.8 us whole
// against 11.0 us split, 64: 25.2 against 19.5, 128: 26.5 against 32.6, 256:
// 29.2 against 35.9; from 384 transforms on the split kernels win again (1792:
// 197 us against 256 us). So batches of NTT_WHOLE_MIN_JOBS = 96 to
// NTT_WHOLE_MAX_JOBS = 256 (the CU count) use the first, the others the second
// (the segment-sum epilogue exists in the first only).
// (Those figures are of Shoup products on the 60-bit limbs. With the folded
// products the 256-transform batch of 64 polynomials measured 35.7 us with the
// copy before it on the whole kernel and 40.0 on the split ones, one stream by
// itself: the same side.)
#include "ntt_kernels.h"

namespace th {

constexpr int NTT_WHOLE_MAX_LOGN = 14;
#ifndef NTT_WHOLE_MAX_JOBS
#define NTT_WHOLE_MAX_JOBS 256
#endif
#ifndef NTT_WHOLE_MIN_JOBS
#define NTT_WHOLE_MIN_JOBS 96
#endif

// Sizes and batches the whole-polynomial kernel cannot serve.
static bool whole_unavailable(int logn, uint32_t njobs) {
  return logn >= NTT_SPLIT_MIN_LOGN && (logn > NTT_WHOLE_MAX_LOGN || njobs > NTT_WHOLE_MAX_JOBS);
}
static bool use_split(int logn, uint32_t njobs) {
  return whole_unavailable(logn, njobs) || (logn >= NTT_SPLIT_MIN_LOGN && njobs < NTT_WHOLE_MIN_JOBS);
}

hipError_t launch_rescale(int logn, const NttArgs& inv, uint32_t ninv, const NttArgs& fwd, uint32_t nfwd,
                          hipStream_t s) {
  if (ninv == 0) return hipSuccess;
  if (use_split(logn, nfwd) && inv.jobs && fwd.jobs && nfwd % ninv == 0 && inv.store == NTT_STORE_NONE &&
      fwd.load == NTT_LOAD_REDUCE)
    return inv.lc.pm ? launch_rescale_split<PmArith>(logn, inv, ninv, fwd, nfwd / ninv, s)
                     : launch_rescale_split<IntArith>(logn, inv, ninv, fwd, nfwd / ninv, s);
  hipError_t e = launch_ntt(logn, true, inv, ninv, s);
  if (e != hipSuccess) return e;
  return launch_ntt(logn, false, fwd, nfwd, s);
}

bool encrypt_limbs_supported(int logn) { return logn >= NTT_SPLIT_MIN_LOGN && logn <= NTT_MAX_LOGN; }

hipError_t launch_encrypt(int logn, const NttArgs& a, uint32_t ninputs, uint32_t L, uint32_t limb_mask,
                          const EncDot& dot, const uint64_t* pkp, uint64_t* cts, bool* combined, hipStream_t s) {
  *combined = false;
  if (ninputs == 0) return hipSuccess;
  const uint32_t nl = (uint32_t)__builtin_popcount(limb_mask);
  if (nl == 0 || limb_mask >> L || (dot.mask & ~limb_mask)) return hipErrorInvalidValue;
  // the split kernels also serve limb subsets and D (k_encrypt_combine forms every limb of c0 and c1)
  const bool split = use_split(logn, ninputs * 3 * nl) || ((nl != L || dot.mask) && encrypt_limbs_supported(logn));
  if (split && a.jobs && a.load == NTT_LOAD_ENC && a.store == NTT_STORE_NONE) {
    *combined = true;
    return a.lc.pm ? launch_encrypt_split<PmArith>(logn, a, ninputs, L, limb_mask, dot, pkp, cts, s)
                   : launch_encrypt_split<IntArith>(logn, a, ninputs, L, limb_mask, dot, pkp, cts, s);
  }
  if (nl != L || dot.mask) return hipErrorInvalidValue;  // k_encrypt_combine forms every limb, no D
  return launch_ntt(logn, false, a, ninputs * 3 * L, s);
}

hipError_t launch_ntt(int logn, bool inverse, const NttArgs& a, uint32_t njobs, hipStream_t s) {
  if (njobs == 0) return hipSuccess;
  const bool segsum = a.jobs && a.store == NTT_STORE_SEGSUM;
  if (segsum && (!inverse || whole_unavailable(logn, njobs) || logn > NTT_WHOLE_MAX_LOGN || a.cols < 1 ||
                 a.cols > NTT_SEGSUM_FUSED_MAX_COLS))
    return hipErrorInvalidValue;  // the segment-sum epilogue exists in the whole-polynomial inverse only
  if (!segsum && use_split(logn, njobs))
    return a.lc.pm ? launch_ntt_split<PmArith>(logn, inverse, a, njobs, s)
                   : launch_ntt_split<IntArith>(logn, inverse, a, njobs, s);
  return a.lc.pm ? launch_ntt_whole<PmArith>(logn, inverse, a, njobs, s)
                 : launch_ntt_whole<IntArith>(logn, inverse, a, njobs, s);
}

hipError_t launch_rescale_decrypt(int logn, const RescaleDecryptArgs& a, uint32_t njobs, hipStream_t s) {
  return a.lc.pm ? launch_rescale_decrypt_whole<PmArith>(logn, a, njobs, s)
                 : launch_rescale_decrypt_whole<IntArith>(logn, a, njobs, s);
}

hipError_t launch_rescale_decrypt_split(int logn, const NttArgs& inv, const RescaleDecryptArgs& a, uint32_t nb,
                                        double* partials, hipStream_t s) {
  return a.lc.pm ? launch_rd_split<PmArith>(logn, inv, a, nb, partials, s)
                 : launch_rd_split<IntArith>(logn, inv, a, nb, partials, s);
}

hipError_t launch_decrypt_sums_split(int logn, const NttArgs& row, const RescaleDecryptArgs& a, uint32_t nb,
                                     double* partials, hipStream_t s) {
  return a.lc.pm ? launch_dec_split<PmArith>(logn, row, a, nb, partials, s)
                 : launch_dec_split<IntArith>(logn, row, a, nb, partials, s);
}

}  // namespace th
