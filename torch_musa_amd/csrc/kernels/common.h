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

}  // namespace tmq
