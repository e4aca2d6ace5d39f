// Rules on sizes, and the job lists' ring, that need no device: kept apart from
// HIP so that a host program can evaluate them (tests/test_launch_rules.py).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace th {

// Whether a device-to-host copy is waited for by polling the stream (else in
// the runtime). The runtime makes copies of up to 16 KiB with a kernel, whose
// end a query cannot see without a marker of its own: polled, a key's draws
// (4 bytes read back) took 41 us against 34, a ciphertext of 16 KiB 26 against
// 15, 512 segment sums (16 KiB) 100 against 94. Larger copies run on the copy
// engine, whose signal the query reads: a decryption behind a product, 32 KiB
// to 128 KiB, 96 / 105 / 117 us polled against 104 / 113 / 126 at N = 8192 /
// 16384 / 32768. Beyond 256 KiB the copy itself takes the time and the wait
// makes no difference.
constexpr bool poll_download(size_t bytes) { return bytes > (16u << 10) && bytes <= (256u << 10); }

// A transform of N complex values (encoder, decoder) is cut into 2^lp parts of
// N / 2^lp values, one workgroup each, of an eighth as many threads (64 to
// 1024; decodes: decode_threads); the result is the same for any split. From 8 parts on a part stages
// its twiddles in LDS beside its values (fft_part_lds): 4096 values take 72
// KiB, 136 with the twiddles, so at N = 32768 a CU holds one workgroup of 512
// threads; 8192 values take 144 KiB with 1024 threads.
//
// Encodes: parts of at most 4096 values, and more of them (up to 16, of at
// least 1024 values) while the batch makes fewer than 512 workgroups. 672
// encodes of N = 16384 per CryptoMOE token: the token measured 0.656 ms with
// parts of 4096 values against 0.697 ms with 8192, 0.675 ms with 2048 and
// 0.727 ms with 1024.
constexpr uint32_t encode_parts_log(uint32_t logn, uint32_t njobs) {
  uint32_t lp = logn <= 12 ? 0 : logn - 12;
  while (lp < 4 && logn - lp > 10 && njobs * (1u << lp) < 512) ++lp;
  return lp;
}

// Decodes: parts of 4096 values, 8192 at N = 32768, and more of them (up to 16,
// of at least 1024 values) while they are still one workgroup per CU. Batches
// with 4 / 8 / 16 parts each:
//   N = 32768, 64 decodes     92 / 107 / 112 us (CRT 119 / 143 / 145)
//   N = 32768, 256            267 / 307 / 314   (CRT 365 / 444 / 424)
//   N = 32768, 24             69 / 63 / 69      (CRT 85 / 81 / 87)
//   N = 32768, 16             66 / 59 / 59
//   N = 16384, 33             57 / 61 / 65      (CRT 70 / 77 / 83)
//   N = 16384, 16             52 / 49 / 49
constexpr uint32_t DECODE_FILL = 256;  // workgroups: the CU count
constexpr uint32_t decode_parts_log(uint32_t logn, uint32_t njobs) {
  uint32_t lp = logn <= 12 ? 0 : logn == 13 ? 1 : 2;
  while (lp < 4 && logn - lp > 10 && ((uint64_t)njobs << (lp + 1)) <= DECODE_FILL) ++lp;
  return lp;
}

// Threads of a decode's part. A thread converts its residues one after another
// (through 128 bits on the CRT path), so a quarter as many threads as values
// where they find room: in parts of up to 2048 values, and in larger ones while
// a CU has only one of them and no staged twiddles. An eighth / a quarter, CRT:
//   N = 1024, 256 decodes     74.4 / 70.7 us    N = 2048, 256   84.1 / 82.4
//   N = 16384, one            48.6 / 46.4       N = 16384, 64   85.0 / 82.8
//   N = 4096, 255             96.0 / 93.8       N = 8192, 64    66.2 / 64.2
// and where two parts share a CU or twiddles are staged:
//   N = 8192, 256            128.6 / 137.8      N = 16384, 128  112.3 / 122.6
//   N = 32768, 24 (limb 0)    62.7 / 64.5
constexpr uint32_t decode_threads(uint32_t logn, uint32_t lp, uint32_t njobs) {
  const uint32_t M = (1u << logn) >> lp;
  const bool room = M <= 2048 || (lp < 3 && ((uint64_t)njobs << lp) <= DECODE_FILL);
  const uint32_t t = room ? M / 4 : M / 8;
  return t < 64 ? 64 : t > 1024 ? 1024 : t;
}

// Places for short job lists in a ring of `cap` bytes, handed out in turn on
// 256-byte boundaries. A list that does not fit behind the last one starts a
// new lap, for which drain() first waits for everything queued so far: a place
// is never handed out again while a queued kernel may read it.
class SlotRing {
 public:
  explicit constexpr SlotRing(size_t cap) : cap_(cap) {}
  // the offset of a place of `bytes` <= cap bytes
  template <class Drain>
  size_t place(size_t bytes, Drain&& drain) {
    const size_t step = (bytes + 255) & ~(size_t)255;
    if (off_ + step > cap_) {
      drain();
      off_ = 0;
    }
    const size_t at = off_;
    off_ += step;
    return at;
  }

 private:
  size_t cap_, off_ = 0;
};

}  // namespace th
