// Shared helpers of the tmq kernel library (device code for gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>
#include <utility>

#include "tmq.h"

#define TMQ_EXPORT extern "C" __attribute__((visibility("default")))

namespace tmq {

constexpr int kWave = 64;  // CDNA wavefront width

static inline hipStream_t as_stream(tmq_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// Status of the launch that was just enqueued (no device synchronisation).
static inline int launch_status() {
  return hipGetLastError() == hipSuccess ? TMQ_OK : TMQ_ERR_LAUNCH;
}

// A kernel onto a stream: one call of the runtime.  The triple-chevron form is three -- the launch shape pushed, popped
// again by the kernel's host stub, and this one -- at 2.48 us against 2.33 us of host time, of the 3.6 ... 4.1 us that an
// operator takes.  launch_status() has the outcome.
template <class... P, class... A>
static inline void enqueue(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A&&... args) {
  // what the kernel's parameters are; braces: an argument that one of them is too narrow for does not compile
  std::tuple<P...> values{P{std::forward<A>(args)}...};
  std::apply(
      [&](P&... v) {
        void* pointers[] = {const_cast<void*>(static_cast<const void*>(&v))..., nullptr};
        (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, lds, stream);
      },
      values);
}

static inline bool aligned(const void* p, uintptr_t a) {
  return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}

__host__ __device__ static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
__host__ __device__ static inline int64_t round_up(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Stores that the L2 passes on as it takes them (device scope).  Lines that a kernel leaves dirty in the eight L2s, 4 MB
// each, are written back between its last instruction and the next kernel's first, with nothing to run beside it: a layer
// that writes 4 to 16 MB pays 1 to 4 us for that (3 -> 64 channels, 7 x 7 stride 2, [32, 3, 224, 224]: 13.3 us inside the
// kernel, 18.8 to the next one's start; with these stores 14.8).  The readers that follow find the bytes in the last-level
// cache either way; where they are few and the reader's blocks run on the XCDs that wrote them (a dequantizer behind up to
// 1 MB) the reader is 0.1 to 0.3 us slower, other readers are not: the blocks of a residual network over 1 to 16 images are
// 0 to 9 % faster throughout.
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
