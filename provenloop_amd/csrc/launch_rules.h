// Rules on sizes that need no device, kept apart from HIP so that a host
// program can evaluate them (tests/test_launch_rules.py).
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

}  // namespace th
