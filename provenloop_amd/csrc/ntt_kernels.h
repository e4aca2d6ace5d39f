// Launchers of the transform kernels for one arithmetic above 2^41 (BIG:
// PmArith or IntArith), instantiated by ntt.hip and ntt_split.hip; callers go
// through the launch_* functions of th_internal.h (ntt_launch.hip).
#pragma once
#include "th_internal.h"

namespace th {

struct IntArith;
struct PmArith;

template <class BIG>
hipError_t launch_ntt_whole(int logn, bool inverse, const NttArgs& a, uint32_t njobs, hipStream_t s);
template <class BIG>
hipError_t launch_rescale_decrypt_whole(int logn, const RescaleDecryptArgs& a, uint32_t njobs, hipStream_t s);
template <class BIG>
hipError_t launch_ntt_split(int logn, bool inverse, const NttArgs& a, uint32_t njobs, hipStream_t s);
template <class BIG>
hipError_t launch_rescale_split(int logn, const NttArgs& inv, uint32_t ninv, const NttArgs& fwd, uint32_t nf,
                                hipStream_t s);
template <class BIG>
hipError_t launch_encrypt_split(int logn, const NttArgs& a, uint32_t ninputs, uint32_t L, uint32_t limb_mask,
                                const EncDot& dot, const uint64_t* pkp, uint64_t* cts, hipStream_t s);
template <class BIG>
hipError_t launch_rd_split(int logn, const NttArgs& inv, const RescaleDecryptArgs& a, uint32_t nb, double* partials,
                           hipStream_t s);
template <class BIG>
hipError_t launch_dec_split(int logn, const NttArgs& row, const RescaleDecryptArgs& a, uint32_t nb, double* partials,
                            hipStream_t s);

}  // namespace th
