// Where a 16-byte read near the end of a tensor goes, for host and device code.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace tmq {

// The 16 bytes at offset `o` (0 <= o < bytes, bytes >= 16) of a tensor of `bytes` bytes: read at `at`, then
// moved down by `shift` bytes (0 ... 15).  At the tensor's end the read starts earlier, so that nothing
// behind it is touched.  Compared in 64 bits: only the bounded difference is narrowed, the distance to the
// tensor's end does not fit 32 bits where more than 2 GiB lie behind `o`.
struct TailRead {
  int64_t at;
  int shift;
};
__host__ __device__ inline TailRead tail_read16(int64_t o, int64_t bytes) {
  const int64_t last = bytes - 16;
  return o > last ? TailRead{last, static_cast<int>(o - last)} : TailRead{o, 0};
}

}  // namespace tmq
