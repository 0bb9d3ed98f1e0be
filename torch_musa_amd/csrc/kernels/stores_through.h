// Byte stores past the L2 (device code for gfx950 only).
#pragma once

#include "common.h"

namespace tmq {

// Stores that the L2 passes on as it takes them (device scope).  Lines that a kernel leaves dirty in the eight L2s, 4 MB
// each, are written back between its last instruction and the next kernel's first, with nothing to run beside it: a layer
// that writes 4 to 16 MB pays 1 to 4 us for that (3 -> 64 channels, 7 x 7 stride 2, [32, 3, 224, 224]: 13.3 us inside the
// kernel, 18.8 to the next one's start; with these stores 14.8).  The readers that follow find the bytes in the last-level
// cache either way.  Where fewer of them than the L2s hold go to blocks on the XCDs that wrote them (an elementwise kernel
// behind another) the reader loses what the writer gains; other readers do not: the blocks of a residual network over 1 to
// 16 images are 0 to 9 % faster throughout.
typedef uint32_t v4u_global __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void st16_through(void* p, v4i v) {  // any alignment
  __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) v4u_global*)(p),
                                     __builtin_bit_cast(v4u_global, v), "agent");
}
__device__ __forceinline__ void st8_through(void* p, uint64_t v) {  // on the 8-byte grid
  __hip_atomic_store(static_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st4_through(void* p, uint32_t v) {  // on the 4-byte grid
  __hip_atomic_store(static_cast<uint32_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace tmq
