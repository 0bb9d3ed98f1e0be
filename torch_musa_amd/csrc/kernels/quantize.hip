// Affine quantize / dequantize / range calibration for gfx950.
//
// All of these are HBM-streaming kernels: 5 bytes of traffic per element for
// quantize and dequantize (4 + 1), 4 for min/max.  Every wave instruction
// touches one dense run of memory: a lane moves 16 bytes of fp32 and the
// matching 4 bytes of codes, so loads and stores are both fully coalesced, and
// each thread keeps several independent 16-byte accesses in flight.
//
// Numerics follow PyTorch's CPU quantizer (fbgemm/QuantUtils.h:67-101,155-158):
// multiply by the fp32 reciprocal of the fp32 scale, round half to even, add
// the zero point, clamp.  Compiled with -ffp-contract=off.
#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

#include "common.h"
#include "device_info.h"
#include "host_report.h"
#include "qparams.h"
#include "quantize_held.h"
#include "stores_through.h"

namespace tmq {
namespace {

constexpr int kThreads = 256;
constexpr int kUnroll = 8;    // independent 16-byte loads per thread, min/max pass
// quantize / dequantize: 2 accesses per thread measured fastest on MI355X at
// 2**28 elements (6.7 and 7.2 TB/s of algorithmic traffic; 8 per thread: 6.0 / 5.3)
constexpr int kUnrollQD = 2;

// FUSED = false: q = clamp(rne(fl(x * inv)) + zp), the arithmetic of
// quantize_per_tensor.  FUSED = true: q = clamp(rne(fl(x * inv + zp))), one
// rounding of product and zero point together, which is how PyTorch's CPU
// quantized::linear_dynamic quantizes its activations while it packs them
// (fbgemm PackAWithQuantRowOffset: fmadd, clip, cvtps); the two differ for
// about one value in 10^5 whose product lies next to a half.
template <bool SIGNED, bool FUSED = false>
__device__ __forceinline__ int quantize_one(float x, float inv, float zp_f) {
  constexpr float lo = SIGNED ? -128.f : 0.f;
  constexpr float hi = SIGNED ? 127.f : 255.f;
  float r;
  if constexpr (FUSED) {
    r = __builtin_rintf(__builtin_fmaf(x, inv, zp_f));
  } else {
    float t = x * inv;
    r = __builtin_rintf(t);  // v_rndne_f32: ties to even
    // zp_f and every in-range r are small integers, so the sum is exact whenever
    // it can land inside [lo, hi]; larger magnitudes clamp either way.
    r = r + zp_f;
  }
  r = fminf(fmaxf(r, lo), hi);
  return static_cast<int>(r);
}

// Four values into one word.  v_cvt_pk_u8_f32 rounds to nearest even, saturates to [0, 255] (NaN -> 0,
// as the clamp of quantize_one has it) and writes its byte into the word: it stands for the clamp, the
// conversion and the packing -- and, where product and zero point are rounded together, for the rounding
// as well.  Signed bytes are the unsigned ones for a zero point 128 higher with the sign bits flipped.
template <bool SIGNED, bool FUSED = false>
__device__ __forceinline__ uint32_t quantize_four(v4f v, float inv, float zp_f) {
  const float zp_u = SIGNED ? zp_f + 128.f : zp_f;
  uint32_t packed = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float r;
    if constexpr (FUSED && SIGNED)  // (the one rounding of product and zero point is that of the signed zero point)
      r = __builtin_rintf(__builtin_fmaf(v[j], inv, zp_f)) + 128.f;
    else if constexpr (FUSED)
      r = __builtin_fmaf(v[j], inv, zp_u);
    else
      r = __builtin_rintf(v[j] * inv) + zp_u;
    packed = __builtin_amdgcn_cvt_pk_u8_f32(r, j, packed);
  }
  return SIGNED ? packed ^ 0x80808080u : packed;
}

template <bool SIGNED>
__device__ __forceinline__ float dequantize_one(uint32_t byte, int zp, float scale) {
  int v = SIGNED ? static_cast<int>(static_cast<int8_t>(byte)) : static_cast<int>(byte);
  return scale * static_cast<float>(v - zp);
}

// Four bytes of one word.  Byte to float is one instruction (v_cvt_f32_ubyte0..3); the zero point is
// subtracted in fp32, where both terms are small integers and the difference is the exact float(q - zp);
// signed bytes are read as unsigned with the sign bits flipped, against a zero point 128 higher.
template <bool SIGNED>
__device__ __forceinline__ v4f dequantize_four(uint32_t w, int zp, float scale) {
  const uint32_t u = SIGNED ? w ^ 0x80808080u : w;
  const float zp_f = static_cast<float>(SIGNED ? zp + 128 : zp);
  v4f r;
  r.x = scale * (static_cast<float>(u & 0xffu) - zp_f);
  r.y = scale * (static_cast<float>((u >> 8) & 0xffu) - zp_f);
  r.z = scale * (static_cast<float>((u >> 16) & 0xffu) - zp_f);
  r.w = scale * (static_cast<float>(u >> 24) - zp_f);
  return r;
}

// Where the scale / zero point come from: kernel arguments, or device memory
// written earlier on the stream by choose_qparams_kernel.
struct QParamsArg {
  float inv;
  float zp_f;
  const tmq_qparams* dev;
};

__device__ __forceinline__ void resolve(const QParamsArg& a, float& inv, float& zp_f) {
  if (a.dev != nullptr) {
    inv = 1.0f / static_cast<float>(a.dev->scale);  // IEEE division
    zp_f = static_cast<float>(a.dev->zero_point);
  } else {
    inv = a.inv;
    zp_f = a.zp_f;
  }
}

// x4/q4 view the first 4*n4 elements; the block with index 0 also converts the
// n - 4*n4 (< 4) trailing elements one by one.
// The fp32 input is read once and never again: non-temporal loads keep it out of
// the caches.  The codes are written with ordinary stores, so a consumer that
// follows on the stream (dequantize, a GEMM) finds them in the last-level cache --
// unless there are more of them than that cache has bytes, 256 Mi: then they leave
// with non-temporal stores as well (kQStream).  Quantize and dequantize of 2**28
// values, us, non-temporal | ordinary: 407 | 375 with one buffer of codes call after
// call, 405 | 386 with three in turn (2**27: 204 | 195; the quantizer by itself,
// three buffers: 199 | 208); of 1.5 * 2**28: 606 | 640, 2**29: 808 | 853.
// Blocks of two waves, as for the dequantizer below: of 128 / 256 / 512 threads with two
// or four accesses each, two waves x two accesses moved 2**28 elements fastest (213 us
// against 219-225 us in one run).
constexpr int kQThreads = 128;

constexpr int64_t kStreamOutCodes = int64_t{1} << 28;  // the last-level cache, in bytes
enum QStore { kQCached, kQThrough, kQStream };
template <bool SIGNED, bool FUSED = false, int STORE = kQCached>
__global__ __launch_bounds__(kQThreads) void quantize_vec_kernel(
    const v4f* __restrict__ x4, uint32_t* __restrict__ q4, int64_t n4,
    const float* __restrict__ x, uint8_t* __restrict__ q, int64_t n, QParamsArg qp) {
  float inv, zp_f;
  resolve(qp, inv, zp_f);
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kQThreads * kUnrollQD) + threadIdx.x;
  v4f v[kUnrollQD];
  if (base - threadIdx.x + kQThreads * kUnrollQD <= n4) {
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) v[u] = __builtin_nontemporal_load(&x4[base + u * kQThreads]);
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) {
      const uint32_t codes = quantize_four<SIGNED, FUSED>(v[u], inv, zp_f);
      if constexpr (STORE == kQStream) __builtin_nontemporal_store(codes, &q4[base + u * kQThreads]);
      else if constexpr (STORE == kQThrough) st4_through(&q4[base + u * kQThreads], codes);
      else q4[base + u * kQThreads] = codes;
    }
  } else {
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) {
      const int64_t i = base + u * kQThreads;
      if (i < n4) v[u] = x4[i];
    }
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) {
      const int64_t i = base + u * kQThreads;
      if (i < n4) q4[i] = quantize_four<SIGNED, FUSED>(v[u], inv, zp_f);
    }
  }
  if (blockIdx.x == 0) {
    const int64_t i = 4 * n4 + threadIdx.x;
    if (i < n) q[i] = static_cast<uint8_t>(quantize_one<SIGNED, FUSED>(x[i], inv, zp_f));
  }
}

// Fallback for pointers that are not 16-byte (x) / 4-byte (q) aligned.
template <bool SIGNED, bool FUSED = false>
__global__ __launch_bounds__(kThreads) void quantize_scalar_kernel(
    const float* __restrict__ x, uint8_t* __restrict__ q, int64_t n, QParamsArg qp) {
  float inv, zp_f;
  resolve(qp, inv, zp_f);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride)
    q[i] = static_cast<uint8_t>(quantize_one<SIGNED, FUSED>(x[i], inv, zp_f));
}

// The codes are read with ordinary loads (they are small and usually still in
// the last-level cache from the kernel that produced them); the fp32 output is
// four times larger and streams out with non-temporal stores so that it does
// not evict them.
// Blocks of two waves: the kernel is bound by the mix of reads and writes at memory (6.5 TB/s of both, 7.1 where the codes
// are still in the last-level cache; a fill of 1 GiB 6.6), and of the
// block sizes 64 ... 1024 two waves with two accesses per thread sustained the
// most over 2**28 elements (204.8 us against 210-240 us for the others).  Stores past the L2s (sc1 nt) with four waves
// take 3 to 6 % off this kernel alone and add up to a fifth to the quantizer beside it; persistent blocks are behind.
constexpr int kDqThreads = 128;

template <bool SIGNED>
__global__ __launch_bounds__(kDqThreads) void dequantize_vec_kernel(
    const uint32_t* __restrict__ q4, v4f* __restrict__ r4, int64_t n4,
    const uint8_t* __restrict__ q, float* __restrict__ r, int64_t n, float scale, int zp) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kDqThreads * kUnrollQD) + threadIdx.x;
  uint32_t w[kUnrollQD];
  if (base - threadIdx.x + kDqThreads * kUnrollQD <= n4) {
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) w[u] = q4[base + u * kDqThreads];
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u)
      __builtin_nontemporal_store(dequantize_four<SIGNED>(w[u], zp, scale), &r4[base + u * kDqThreads]);
  } else {
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) {
      const int64_t i = base + u * kDqThreads;
      if (i < n4) w[u] = q4[i];
    }
#pragma unroll
    for (int u = 0; u < kUnrollQD; ++u) {
      const int64_t i = base + u * kDqThreads;
      if (i < n4) r4[i] = dequantize_four<SIGNED>(w[u], zp, scale);
    }
  }
  if (blockIdx.x == 0) {
    const int64_t i = 4 * n4 + threadIdx.x;
    if (i < n) r[i] = dequantize_one<SIGNED>(q[i], zp, scale);
  }
}

template <bool SIGNED>
__global__ __launch_bounds__(kThreads) void dequantize_scalar_kernel(
    const uint8_t* __restrict__ q, float* __restrict__ r, int64_t n, float scale, int zp) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride)
    r[i] = dequantize_one<SIGNED>(q[i], zp, scale);
}

// ---------------------------------------------------------------------------
// min / max: persistent grid, 16-byte loads, wavefront butterfly reduction,
// one {min,max} pair per block, then a one-block second stage.
// ---------------------------------------------------------------------------
constexpr int kMinMaxMaxBlocks = 2048;  // (1024 ... 4096 blocks and 4 ... 8 loads per thread measure alike)

__device__ __forceinline__ void wave_minmax(float& mn, float& mx) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
  }
}

__device__ __forceinline__ void block_minmax_store(float mn, float mx, float* out) {
  __shared__ float s_mn[kThreads / kWave];
  __shared__ float s_mx[kThreads / kWave];
  wave_minmax(mn, mx);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  if (lane == 0) {
    s_mn[wave] = mn;
    s_mx[wave] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kThreads / kWave; ++w) {
      mn = fminf(mn, s_mn[w]);
      mx = fmaxf(mx, s_mx[w]);
    }
    out[0] = mn;
    out[1] = mx;
  }
}

// Blocks of the range passes that have written their partial pair, by report: the last one wraps the
// count back to 0 (and the memory starts as 0), a report belongs to one call at a time.
__device__ unsigned int g_range_arrivals[TMQ_HOST_REPORTS];

// KEEP: ordinary loads instead of non-temporal ones, for an input that a second pass on
// the stream reads again while the last-level cache still holds it.
// With a report, the last block to arrive reduces the partial pairs and tells the host the
// range, one launch earlier than the pass behind this one could.
template <bool KEEP = false>
__global__ __launch_bounds__(kThreads) void minmax_partial_kernel(
    const v4f* __restrict__ x4, int64_t n4, const float* __restrict__ x, int64_t head,
    int64_t n, float* __restrict__ partials, RangeReport report) {
  auto ld = [](const v4f* p) { return KEEP ? *p : __builtin_nontemporal_load(p); };
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  const int64_t step = static_cast<int64_t>(gridDim.x) * (kThreads * kUnroll);
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * (kThreads * kUnroll) + threadIdx.x;
       base - threadIdx.x < n4; base += step) {
    v4f v[kUnroll];
    if (base - threadIdx.x + kThreads * kUnroll <= n4) {
      // a whole chunk: unconditional loads, all in flight before the first comparison
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) v[u] = ld(&x4[base + u * kThreads]);
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        mn = fminf(fminf(mn, v[u].x), fminf(v[u].y, fminf(v[u].z, v[u].w)));
        mx = fmaxf(fmaxf(mx, v[u].x), fmaxf(v[u].y, fmaxf(v[u].z, v[u].w)));
      }
      continue;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t i = base + u * kThreads;
      if (i < n4) v[u] = ld(&x4[i]);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int64_t i = base + u * kThreads;
      if (i < n4) {
        mn = fminf(fminf(mn, v[u].x), fminf(v[u].y, fminf(v[u].z, v[u].w)));
        mx = fmaxf(fmaxf(mx, v[u].x), fmaxf(v[u].y, fmaxf(v[u].z, v[u].w)));
      }
    }
  }
  if (blockIdx.x == 0) {
    // elements before the first 16-byte boundary and after the last full group
    const int64_t tail0 = head + 4 * n4;
    const int64_t extra = head + (n - tail0);
    for (int64_t j = threadIdx.x; j < extra; j += kThreads) {
      const float v = j < head ? x[j] : x[tail0 + (j - head)];
      mn = fminf(mn, v);
      mx = fmaxf(mx, v);
    }
  }
  if (report.to == nullptr) {
    block_minmax_store(mn, mx, partials + 2 * blockIdx.x);
    return;
  }
  __shared__ bool s_last;
  __shared__ float s_mm[2];
  block_minmax_store(mn, mx, s_mm);
  if (threadIdx.x == 0) {
    // The pair goes out as one atomic exchange and the block arrives once the exchange has
    // answered, i.e. has been done where every XCD sees it.  (A release fence would write back
    // the L2 instead, which is full of whatever ran before: 40 -> 62 us at [4877, 3648].)
    const uint64_t pair = (static_cast<uint64_t>(__builtin_bit_cast(uint32_t, s_mm[1])) << 32) |
                          __builtin_bit_cast(uint32_t, s_mm[0]);
    const uint64_t before = __hip_atomic_exchange(reinterpret_cast<uint64_t*>(partials) + blockIdx.x, pair,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::"v"(before) : "memory");  // (waits for the answer)
    const unsigned int last = gridDim.x - 1;
    const bool is_last = atomicInc(&g_range_arrivals[report.slot], last) == last;
    // The other blocks' pairs are read behind the count that says they are there: the barrier hands this
    // acquire on to the block's other waves.  (Later loads find no older copy in a cache; nothing is written back.)
    if (is_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    s_last = is_last;
  }
  __syncthreads();
  if (!s_last) return;
  mn = std::numeric_limits<float>::infinity();
  mx = -std::numeric_limits<float>::infinity();
  for (unsigned i = threadIdx.x; i < gridDim.x; i += kThreads) {
    const uint64_t pair = __hip_atomic_load(reinterpret_cast<uint64_t*>(partials) + i, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
    mn = fminf(mn, __builtin_bit_cast(float, static_cast<uint32_t>(pair)));
    mx = fmaxf(mx, __builtin_bit_cast(float, static_cast<uint32_t>(pair >> 32)));
  }
  block_minmax_store(mn, mx, s_mm);
  if (threadIdx.x == 0) report_range(report, s_mm[0], s_mm[1]);
}

__global__ __launch_bounds__(kThreads) void minmax_final_kernel(
    const float* __restrict__ partials, int count, float* __restrict__ out) {
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  for (int i = threadIdx.x; i < count; i += kThreads) {
    mn = fminf(mn, partials[2 * i]);
    mx = fmaxf(mx, partials[2 * i + 1]);
  }
  block_minmax_store(mn, mx, out);
}

__global__ void choose_qparams_kernel(const float* __restrict__ minmax, int qmin, int qmax,
                                      int reduce_range, tmq_qparams* __restrict__ out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    double s;
    int32_t z;
    choose_qparams(minmax[0], minmax[1], qmin, qmax, reduce_range != 0, &s, &z);
    out->scale = s;
    out->zero_point = z;
    out->reserved = 0;
  }
}

// Last stage of the min/max reduction and ChooseQuantizationParams in one block.
__global__ __launch_bounds__(kThreads) void minmax_final_choose_kernel(
    const float* __restrict__ partials, int count, int qmin, int qmax, int reduce_range,
    tmq_qparams* __restrict__ out, RangeReport report) {
  __shared__ float s_mm[2];
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  for (int i = threadIdx.x; i < count; i += kThreads) {
    mn = fminf(mn, partials[2 * i]);
    mx = fmaxf(mx, partials[2 * i + 1]);
  }
  block_minmax_store(mn, mx, s_mm);
  if (threadIdx.x == 0) {
    double s;
    int32_t z;
    choose_qparams(s_mm[0], s_mm[1], qmin, qmax, reduce_range != 0, &s, &z);
    out->scale = s;
    out->zero_point = z;
    out->reserved = 0;
    report_range(report, s_mm[0], s_mm[1]);
  }
}

// Second launch of a dynamic quantization that takes two (quantize_held.h has the one that takes one, which a
// captured stream cannot run): every block first finishes the range
// reduction for itself -- the partial {min, max} pairs of the pass before it (at most
// kDynPartials of them, 4 KB from the L2s), ChooseQuantizationParams in one thread --
// while the loads of its first elements are already in flight, then quantizes its
// share of the input in a grid-stride loop with the next chunk requested before the
// current one is converted.  Block 0 also publishes the parameters.  This replaces a
// one-block launch between the two passes (5 us of a 32 us chain at 2**24 elements:
// launch, 16 KB through one block, the double-precision divisions) by a few hundred
// cycles under each block's first loads.  Same arithmetic in the same order as the
// three launches: min and max do not depend on the order of the reduction.
constexpr int kDynPartials = 512;
constexpr int kDynQBlocks = 2048;
// Up to here the range pass itself reports the range (see minmax_partial_kernel): the host is what
// such a call waits for.  Above, the quantizer runs long enough for the host to hear from its first
// block in time, and the range pass is spared its last block's extra round of reads.
constexpr int64_t kDynEarlyMax = int64_t{1} << 21;
constexpr int64_t kDynKeepMax = int64_t{1} << 25;  // 128 MiB of fp32: half the last-level cache
template <bool SIGNED, bool FUSED>
__global__ __launch_bounds__(kThreads) void quantize_after_minmax_kernel(
    const v4f* __restrict__ x4, uint32_t* __restrict__ q4, int64_t n4, const float* __restrict__ x,
    uint8_t* __restrict__ q, int64_t n, const float* __restrict__ partials, int count, int qmin, int qmax,
    int reduce_range, tmq_qparams* __restrict__ out, RangeReport report) {
  __shared__ float s_mm[2];
  __shared__ float s_inv, s_zp;
  constexpr int U = kUnrollQD;
  const int64_t step = static_cast<int64_t>(gridDim.x) * (kThreads * U);
  int64_t base = static_cast<int64_t>(blockIdx.x) * (kThreads * U) + threadIdx.x;
  // (loads are unconditional -- indices clamped into the input -- so that they can be
  // counted: a load under a condition would be waited for before anything else is requested)
  auto request = [&](int64_t b, v4f(&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = b + u * kThreads;
      v[u] = x4[i < n4 ? i : (n4 > 0 ? n4 - 1 : 0)];
    }
  };
  v4f cur[U], nxt[U];
  if (n4 > 0) request(base, cur);
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  for (int i = threadIdx.x; i < count; i += kThreads) {
    const float2 p = *reinterpret_cast<const float2*>(partials + 2 * i);
    mn = fminf(mn, p.x);
    mx = fmaxf(mx, p.y);
  }
  block_minmax_store(mn, mx, s_mm);  // (ends with thread 0 holding the block's result)
  if (threadIdx.x == 0) {
    double sc;
    int32_t z;
    choose_qparams(s_mm[0], s_mm[1], qmin, qmax, reduce_range != 0, &sc, &z);
    s_inv = 1.0f / static_cast<float>(sc);  // IEEE division, as resolve()
    s_zp = static_cast<float>(z);
    if (blockIdx.x == 0) {
      report_range(report, s_mm[0], s_mm[1]);
      out->scale = sc;
      out->zero_point = z;
      out->reserved = 0;
    }
  }
  __syncthreads();
  const float inv = s_inv, zp_f = s_zp;
  for (; base - threadIdx.x < n4; base += step) {
    const bool more = base - threadIdx.x + step < n4;
    if (more) request(base + step, nxt);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = base + u * kThreads;
      if (i < n4) q4[i] = quantize_four<SIGNED, FUSED>(cur[u], inv, zp_f);
    }
    if (more) {
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = nxt[u];
    }
  }
  if (blockIdx.x == 0) {
    const int64_t i = 4 * n4 + threadIdx.x;
    if (i < n) q[i] = static_cast<uint8_t>(quantize_one<SIGNED, FUSED>(x[i], inv, zp_f));
  }
}

// The same for rows that the product behind it wants on the 16-byte grid: `M` rows of K values
// -> rows of `pitch` codes (a multiple of 16, less than 16 over K), a word of four codes per lane.
// The codes behind a row's end are whatever the last values give; they meet zero weights.
template <bool SIGNED, bool FUSED>
__global__ __launch_bounds__(kThreads) void quantize_rows_after_minmax_kernel(
    const float* __restrict__ x, uint32_t* __restrict__ q4, int64_t M, int32_t K, int32_t pitch4,
    const float* __restrict__ partials, int count, int qmin, int qmax, int reduce_range, tmq_qparams* __restrict__ out) {
  __shared__ float s_mm[2];
  __shared__ float s_inv, s_zp;
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  for (int i = threadIdx.x; i < count; i += kThreads) {
    const float2 p = *reinterpret_cast<const float2*>(partials + 2 * i);
    mn = fminf(mn, p.x);
    mx = fmaxf(mx, p.y);
  }
  block_minmax_store(mn, mx, s_mm);
  if (threadIdx.x == 0) {
    double sc;
    int32_t z;
    choose_qparams(s_mm[0], s_mm[1], qmin, qmax, reduce_range != 0, &sc, &z);
    s_inv = 1.0f / static_cast<float>(sc);  // IEEE division, as resolve()
    s_zp = static_cast<float>(z);
    if (blockIdx.x == 0) {
      out->scale = sc;
      out->zero_point = z;
      out->reserved = 0;
    }
  }
  __syncthreads();
  const float inv = s_inv, zp_f = s_zp;
  const int64_t total = M * pitch4, step = static_cast<int64_t>(gridDim.x) * kThreads;
  int64_t g = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int64_t row = g / pitch4;
  int c4 = static_cast<int>(g - row * pitch4);
  const int64_t step_rows = step / pitch4;  // (one division each, not one per word)
  const int step_c4 = static_cast<int>(step - step_rows * pitch4);
  for (; g < total; g += step) {
    const float* src = x + row * K;
    v4f v = {0.f, 0.f, 0.f, 0.f};
    if (4 * c4 + 4 <= K) {
      __builtin_memcpy(&v, src + 4 * c4, 16);
    } else {
      for (int j = 0; 4 * c4 + j < K; ++j) v[j] = src[4 * c4 + j];
    }
    q4[g] = quantize_four<SIGNED, FUSED>(v, inv, zp_f);
    row += step_rows;
    c4 += step_c4;
    if (c4 >= pitch4) {
      c4 -= pitch4;
      ++row;
    }
  }
}

// Dynamic quantization of a small tensor in one launch.  Every block reads the whole input and
// finds the range for itself -- the same lines for all of them, from the L2s -- and converts its
// own 1024 words of four codes; a block converts what it reads at its own position, so nothing is
// read twice by a block.  No block waits for another.  The read bounds it: 96 Ki values are 384 KB
// into every CU, 2.7 us at 64 bytes a clock, about what the launch and the gap between two launches
// cost (a dynamically quantized linear of 55 rows, 704 -> 480: 12.2 -> 8.6 us; of 283 rows, 392 -> 192,
// 111 Ki values: level; quantize and dequantize of 130 x 384 values 16.7 -> 15.6 us, of 581 x 221
// 16.3 -> 17.4 us, hence the limit; above 32 Ki values it only runs where ranges cannot be exchanged, see kHeldAbove).
// Rows: `K` values each, written at a pitch of 4 pitch4 codes (pitch4 = 0: one row, no pitch).  x is read as
// 16 bytes at any 4-byte alignment.
constexpr int kDynRepeatThreads = 1024;
constexpr int64_t kDynRepeatMax = 98304;
template <bool SIGNED, bool FUSED>
__global__ __launch_bounds__(kDynRepeatThreads) void dynamic_quantize_repeat_kernel(
    const float* __restrict__ x, uint8_t* __restrict__ q, int32_t n, int32_t K, int32_t pitch4, int qmin, int qmax,
    int reduce_range, bool words, tmq_qparams* __restrict__ out, RangeReport report) {
  constexpr int kWaves = kDynRepeatThreads / kWave, kAhead = 8;
  __shared__ float s_mn[kWaves], s_mx[kWaves];
  __shared__ float s_inv, s_zp;
  const int t = threadIdx.x, own = static_cast<int>(blockIdx.x);
  struct __attribute__((packed, aligned(4))) Four {
    v4f v;
  };
  // group i of the input: values 4 i ... 4 i + 3; the last one begins where four values are left (some are then
  // seen twice, which no minimum or maximum minds)
  const auto group = [&](int i) { return reinterpret_cast<const Four*>(x + (4 * i + 4 <= n ? 4 * i : n - 4))->v; };
  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  v4f mine = {0.f, 0.f, 0.f, 0.f};
  const int groups = (n + 3) / 4;
  if (n >= 4 && groups <= kDynRepeatThreads) {
    mine = group(t < groups ? t : groups - 1);
    mn = fminf(fminf(mine.x, mine.y), fminf(mine.z, mine.w));
    mx = fmaxf(fmaxf(mine.x, mine.y), fmaxf(mine.z, mine.w));
  } else if (n >= 4) {
    for (int u0 = 0; u0 * kDynRepeatThreads < groups; u0 += kAhead) {
      v4f v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int i = (u0 + u) * kDynRepeatThreads + t;
        v[u] = group(i < groups ? i : groups - 1);
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        mn = fminf(fminf(mn, v[u].x), fminf(v[u].y, fminf(v[u].z, v[u].w)));
        mx = fmaxf(fmaxf(mx, v[u].x), fmaxf(v[u].y, fmaxf(v[u].z, v[u].w)));
        if (u0 + u == own) mine = v[u];
      }
    }
  } else if (t < n) {
    mn = mx = x[t];
  }
  wave_minmax(mn, mx);
  if (t % kWave == 0) {
    s_mn[t / kWave] = mn;
    s_mx[t / kWave] = mx;
  }
  __syncthreads();
  if (t < kWave) {
    mn = t < kWaves ? s_mn[t] : std::numeric_limits<float>::infinity();
    mx = t < kWaves ? s_mx[t] : -std::numeric_limits<float>::infinity();
    wave_minmax(mn, mx);
    if (t == 0) {
      double s;
      int32_t z;
      if (own == 0) report_range(report, mn, mx);
      choose_qparams(mn, mx, qmin, qmax, reduce_range != 0, &s, &z);
      if (own == 0) {
        out->scale = s;
        out->zero_point = z;
        out->reserved = 0;
      }
      s_inv = 1.0f / static_cast<float>(s);  // IEEE division, as in resolve()
      s_zp = static_cast<float>(z);
    }
  }
  __syncthreads();
  const float inv = s_inv, zp_f = s_zp;
  const int g = own * kDynRepeatThreads + t;  // this thread's word
  if (pitch4 == 0) {
    if (4 * g + 4 <= n && words) {
      reinterpret_cast<uint32_t*>(q)[g] = quantize_four<SIGNED, FUSED>(mine, inv, zp_f);
    } else {
      for (int j = 4 * g; j < 4 * g + 4 && j < n; ++j) q[j] = static_cast<uint8_t>(quantize_one<SIGNED, FUSED>(x[j], inv, zp_f));
    }
    return;
  }
  const int row = g / pitch4, c = 4 * (g - row * pitch4);
  if (row * K >= n) return;
  v4f v = {0.f, 0.f, 0.f, 0.f};
  if (c + 4 <= K) {
    v = reinterpret_cast<const Four*>(x + row * K + c)->v;
  } else {
    for (int j = 0; c + j < K; ++j) v[j] = x[row * K + c + j];
  }
  reinterpret_cast<uint32_t*>(q)[g] = quantize_four<SIGNED, FUSED>(v, inv, zp_f);
}
template <class... Args>
int launch_dynamic_repeat(bool q_signed, bool fused, int64_t words, hipStream_t s, Args... args) {
  const dim3 grid(static_cast<unsigned>((words + kDynRepeatThreads - 1) / kDynRepeatThreads)), block(kDynRepeatThreads);
  if (q_signed && fused) enqueue(dynamic_quantize_repeat_kernel<true, true>, grid, block, 0, s, args...);
  else if (q_signed) enqueue(dynamic_quantize_repeat_kernel<true, false>, grid, block, 0, s, args...);
  else if (fused) enqueue(dynamic_quantize_repeat_kernel<false, true>, grid, block, 0, s, args...);
  else enqueue(dynamic_quantize_repeat_kernel<false, false>, grid, block, 0, s, args...);
  return launch_status();
}

// ---------------------------------------------------------------------------
// Per-channel kernels over [outer, C, inner].  One Op per conversion (double or float
// parameters, either direction); which kernel walks the tensor depends on where the
// channels lie:
//   inner == 1 (a channel axis that is the last dimension in memory): pc_cols_kernel,
//     a thread keeps its channels and walks down the rows;
//   inner % 4 == 0, inner >= 64: pc_rows_kernel, the channel is a property of the block;
//   other inner >= 4: pc_flat_kernel, 16-byte accesses over the flat tensor, a group of
//     four lies in at most two channels;
//   inner 2 and 3: pc_element_kernel.
// ---------------------------------------------------------------------------
template <bool SIGNED>
__device__ __forceinline__ float dequantize_pc_one(uint32_t byte, float zp_f, double scale) {
  const int v = SIGNED ? static_cast<int>(static_cast<int8_t>(byte)) : static_cast<int>(byte);
  const float d = static_cast<float>(v) - zp_f;
  return static_cast<float>(static_cast<double>(d) * scale);
}

// Per-channel quantizer with float scales and float zero points
// (qscheme per_channel_affine_float_qparams): q = clamp(lrintf(x * inv + zp)),
// inv = 1 / scale (1 when the scale is 0), r = (float(q) - zp) * scale, all fp32.
template <bool SIGNED>
__device__ __forceinline__ uint32_t quantize_fq_one(float x, float inv, float zp) {
  const float t = x * inv;
  float r = __builtin_rintf(t + zp);
  r = __builtin_amdgcn_fmed3f(r, SIGNED ? -128.f : 0.f, SIGNED ? 127.f : 255.f);
  return static_cast<uint32_t>(static_cast<int>(r)) & 0xffu;
}

template <bool SIGNED>
__device__ __forceinline__ float dequantize_fq_one(uint32_t byte, float zp, float scale) {
  const int v = SIGNED ? static_cast<int>(static_cast<int8_t>(byte)) : static_cast<int>(byte);
  const float d = static_cast<float>(v) - zp;
  return d * scale;
}

// An Op: P, the parameters of a channel; load4 / load1, conv4 (four values of up to four
// channels), conv1, put4 / put1; zp_outside, the range check of a channel's zero point.
template <bool SIGNED>
struct PcQuantize {
  // fp32 -> codes, double scales, int64 zero points
  static constexpr int kAccesses = 4;
  const float* x;
  uint8_t* q;
  const double* scales;
  const int64_t* zps;
  struct P { float inv, zp; };
  using In4 = v4f;
  using In1 = float;
  using Out4 = uint32_t;
  __device__ __forceinline__ P params(int64_t c) const {
    return {1.0f / static_cast<float>(scales[c]), static_cast<float>(zps[c])};
  }
  __device__ __forceinline__ bool zp_outside(int64_t c) const {
    const int64_t z = zps[c];
    return z < (SIGNED ? -128 : 0) || z > (SIGNED ? 127 : 255);
  }
  __device__ __forceinline__ In4 load4(int64_t i) const {
    return __builtin_nontemporal_load(reinterpret_cast<const v4f*>(x + i));
  }
  __device__ __forceinline__ In1 load1(int64_t i) const { return x[i]; }
  __device__ __forceinline__ Out4 conv4(In4 v, const P (&p)[4]) const {
    uint32_t packed = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)  // (as quantize_four)
      packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(v[j] * p[j].inv) + (SIGNED ? p[j].zp + 128.f : p[j].zp), j,
                                              packed);
    return SIGNED ? packed ^ 0x80808080u : packed;
  }
  __device__ __forceinline__ void put4(int64_t i, Out4 v) const { *reinterpret_cast<uint32_t*>(q + i) = v; }
  __device__ __forceinline__ void put1(int64_t i, In1 v, P p) const {
    q[i] = static_cast<uint8_t>(quantize_one<SIGNED>(v, p.inv, p.zp));
  }
};

template <bool SIGNED>
struct PcDequantize {
  // codes -> fp32, double scales, int64 zero points
  static constexpr int kAccesses = 2;
  const uint8_t* q;
  float* r;
  const double* scales;
  const int64_t* zps;
  struct P { double scale; float zp; };
  using In4 = uint32_t;
  using In1 = uint32_t;
  using Out4 = v4f;
  __device__ __forceinline__ P params(int64_t c) const { return {scales[c], static_cast<float>(zps[c])}; }
  __device__ __forceinline__ bool zp_outside(int64_t c) const {
    const int64_t z = zps[c];
    return z < (SIGNED ? -128 : 0) || z > (SIGNED ? 127 : 255);
  }
  __device__ __forceinline__ In4 load4(int64_t i) const { return *reinterpret_cast<const uint32_t*>(q + i); }
  __device__ __forceinline__ In1 load1(int64_t i) const { return q[i]; }
  __device__ __forceinline__ Out4 conv4(In4 w, const P (&p)[4]) const {
    v4f o;
    o.x = dequantize_pc_one<SIGNED>(w & 0xffu, p[0].zp, p[0].scale);
    o.y = dequantize_pc_one<SIGNED>((w >> 8) & 0xffu, p[1].zp, p[1].scale);
    o.z = dequantize_pc_one<SIGNED>((w >> 16) & 0xffu, p[2].zp, p[2].scale);
    o.w = dequantize_pc_one<SIGNED>(w >> 24, p[3].zp, p[3].scale);
    return o;
  }
  __device__ __forceinline__ void put4(int64_t i, Out4 o) const {
    __builtin_nontemporal_store(o, reinterpret_cast<v4f*>(r + i));
  }
  __device__ __forceinline__ void put1(int64_t i, In1 b, P p) const { r[i] = dequantize_pc_one<SIGNED>(b, p.zp, p.scale); }
};

template <bool SIGNED>
struct PcfQuantize {
  // fp32 -> codes, float scales and float zero points
  static constexpr int kAccesses = 4;
  const float* x;
  uint8_t* q;
  const float* scales;
  const float* zps;
  struct P { float inv, zp; };
  using In4 = v4f;
  using In1 = float;
  using Out4 = uint32_t;
  __device__ __forceinline__ P params(int64_t c) const {
    const float sc = scales[c];
    return {sc == 0.f ? 1.0f : 1.0f / sc, zps[c]};
  }
  __device__ __forceinline__ bool zp_outside(int64_t c) const {
    return zps[c] < (SIGNED ? -128.f : 0.f) || zps[c] > (SIGNED ? 127.f : 255.f);
  }
  __device__ __forceinline__ In4 load4(int64_t i) const {
    return __builtin_nontemporal_load(reinterpret_cast<const v4f*>(x + i));
  }
  __device__ __forceinline__ In1 load1(int64_t i) const { return x[i]; }
  __device__ __forceinline__ Out4 conv4(In4 v, const P (&p)[4]) const {
    return quantize_fq_one<SIGNED>(v.x, p[0].inv, p[0].zp) | (quantize_fq_one<SIGNED>(v.y, p[1].inv, p[1].zp) << 8) |
           (quantize_fq_one<SIGNED>(v.z, p[2].inv, p[2].zp) << 16) | (quantize_fq_one<SIGNED>(v.w, p[3].inv, p[3].zp) << 24);
  }
  __device__ __forceinline__ void put4(int64_t i, Out4 v) const { *reinterpret_cast<uint32_t*>(q + i) = v; }
  __device__ __forceinline__ void put1(int64_t i, In1 v, P p) const {
    q[i] = static_cast<uint8_t>(quantize_fq_one<SIGNED>(v, p.inv, p.zp));
  }
};

template <bool SIGNED>
struct PcfDequantize {
  // codes -> fp32, float scales and float zero points
  static constexpr int kAccesses = 2;
  const uint8_t* q;
  float* r;
  const float* scales;
  const float* zps;
  struct P { float scale, zp; };
  using In4 = uint32_t;
  using In1 = uint32_t;
  using Out4 = v4f;
  __device__ __forceinline__ P params(int64_t c) const { return {scales[c], zps[c]}; }
  __device__ __forceinline__ bool zp_outside(int64_t c) const {
    return zps[c] < (SIGNED ? -128.f : 0.f) || zps[c] > (SIGNED ? 127.f : 255.f);
  }
  __device__ __forceinline__ In4 load4(int64_t i) const { return *reinterpret_cast<const uint32_t*>(q + i); }
  __device__ __forceinline__ In1 load1(int64_t i) const { return q[i]; }
  __device__ __forceinline__ Out4 conv4(In4 w, const P (&p)[4]) const {
    v4f o;
    o.x = dequantize_fq_one<SIGNED>(w & 0xffu, p[0].zp, p[0].scale);
    o.y = dequantize_fq_one<SIGNED>((w >> 8) & 0xffu, p[1].zp, p[1].scale);
    o.z = dequantize_fq_one<SIGNED>((w >> 16) & 0xffu, p[2].zp, p[2].scale);
    o.w = dequantize_fq_one<SIGNED>(w >> 24, p[3].zp, p[3].scale);
    return o;
  }
  __device__ __forceinline__ void put4(int64_t i, Out4 o) const {
    __builtin_nontemporal_store(o, reinterpret_cast<v4f*>(r + i));
  }
  __device__ __forceinline__ void put1(int64_t i, In1 b, P p) const { r[i] = dequantize_fq_one<SIGNED>(b, p.zp, p.scale); }
};

// A quantizer whose codes leave past the L2s.
template <class Op>
struct PcThrough : Op {
  explicit PcThrough(const Op& op) : Op(op) {}
  __device__ __forceinline__ void put4(int64_t i, typename Op::Out4 v) const { st4_through(this->q + i, v); }
};

// The range check of the zero points, which the caller has to raise an error for before it
// returns: the first block of the conversion does nothing else, so the answer is out a few
// microseconds after the kernel starts, while the other blocks convert, and the host goes on
// without waiting for them.  (As a chain of its own, two comparisons, their union and a
// reduction read back by the host, it took 16 us of GPU time and left the queue empty.)
struct PcCheck {
  tmq_host_report* report;
  uint32_t ticket;
};
template <class Op>
__device__ __forceinline__ void pc_check_block(const Op& op, int64_t C, const PcCheck& check) {
  int bad = 0;
  if (C <= static_cast<int64_t>(blockDim.x)) {
    bad = op.zp_outside(threadIdx.x < C ? threadIdx.x : C - 1) ? 1 : 0;
  } else {
    // eight requests in flight per thread: one by one, 11008 zero points took as long as the conversion
    // (fp32 [11008, 4096], both directions: 83 -> 69 us)
    constexpr int kAhead = 8;
    for (int64_t c0 = threadIdx.x; c0 < C; c0 += static_cast<int64_t>(blockDim.x) * kAhead) {
      bool out[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int64_t c = c0 + static_cast<int64_t>(u) * blockDim.x;
        out[u] = op.zp_outside(c < C ? c : C - 1);
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) bad |= out[u] ? 1 : 0;
    }
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) report_word(&check.report->word[0], check.ticket, bad != 0 ? 1u : 0u);
}
// This block's index among the converting ones; negative: it was the checking one.
template <class Op>
__device__ __forceinline__ int64_t pc_block(const Op& op, int64_t C, const PcCheck& check) {
  if (check.report == nullptr) return blockIdx.x;
  if (blockIdx.x == 0) pc_check_block(op, C, check);
  return static_cast<int64_t>(blockIdx.x) - 1;
}

constexpr int kPcRowsMinInner = 64;

// pc_rows_kernel: the tensor is `rows` = outer * C rows of `inner` elements; a block takes
// RB = A >> lg_us consecutive rows (A accesses per thread) x one segment of US = 1 << lg_us
// runs of 128 lanes x 4 elements.  Row and channel come from blockIdx with one division per
// block; the parameters of a row are wave-uniform (scalar loads); the element loop has no
// division at all.  Accesses per thread (Op::kAccesses), all in flight before the first
// store: four for the quantizers, two for the dequantizers, in blocks of two waves -- the
// shape the per-tensor kernels settled on as well.  At fp32 [11008, 4096], axis 0, inputs and
// outputs rotating over more bytes than the last-level cache holds: quantize 39.8 us
// (per-tensor kernel on as many elements: 38.4 us), dequantize 37.6 us (35.4 us);
// the dequantizer took 42.2 us with a parameter request per access, each waiting for
// the one before it, 39.4 us with one per row in blocks of four waves x four accesses.
constexpr int kPcThreads = 128;
template <class Op>
__global__ __launch_bounds__(kPcThreads) void pc_rows_kernel(Op op, int64_t rows, int64_t C, int64_t inner,
                                                           int lg_us, uint32_t segs, PcCheck check) {
  constexpr int kPcAccesses = Op::kAccesses, VEC = 4;
  const int64_t block = pc_block(op, C, check);
  if (block < 0) return;
  const uint32_t rg = static_cast<uint32_t>(block) / segs, seg = static_cast<uint32_t>(block) - rg * segs;
  const int us_mask = (1 << lg_us) - 1;
  const int64_t row0 = static_cast<int64_t>(rg) * (kPcAccesses >> lg_us);
  const int64_t c0 = row0 % C;  // once per block, wave-uniform
  const int64_t col0 = (static_cast<int64_t>(seg) << lg_us) * (kPcThreads * VEC) + threadIdx.x * VEC;
  typename Op::In4 held[kPcAccesses];
  bool live[kPcAccesses];
  // a block that lies inside the tensor as a whole (all but the last row group and the
  // last segment of a row) loads and stores without a condition per access
  const bool whole = row0 + (kPcAccesses >> lg_us) <= rows &&
                     ((static_cast<int64_t>(seg) + 1) << lg_us) * (kPcThreads * VEC) <= inner;
  if (whole) {
    // with the number of runs per row as a constant, every index below is one: the
    // parameters of the block's rows are requested together, once per row (not once
    // per access, each request waiting for the one before it)
    auto run = [&](auto lg_tag) {
      constexpr int LG = decltype(lg_tag)::value;
      if constexpr ((1 << LG) <= kPcAccesses) {
        constexpr int kRows = kPcAccesses >> LG, kRuns = 1 << LG;
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
          for (int k = 0; k < kRuns; ++k)
            held[r * kRuns + k] = op.load4((row0 + r) * inner + col0 + static_cast<int64_t>(k) * (kPcThreads * VEC));
        typename Op::P prm[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
          int64_t c = c0 + r;
          while (c >= C) c -= C;   // at most kRows - 1 rows past c0: uniform, a few scalar steps
          prm[r] = op.params(c);
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
          for (int k = 0; k < kRuns; ++k) {
            const int64_t at = (row0 + r) * inner + col0 + static_cast<int64_t>(k) * (kPcThreads * VEC);
            op.put4(at, op.conv4(held[r * kRuns + k], {prm[r], prm[r], prm[r], prm[r]}));
          }
      }
    };
    switch (lg_us) {
      case 0: run(std::integral_constant<int, 0>{}); break;
      case 1: run(std::integral_constant<int, 1>{}); break;
      case 2: run(std::integral_constant<int, 2>{}); break;
      default: run(std::integral_constant<int, 3>{}); break;
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < kPcAccesses; ++u) {
    const int64_t row = row0 + (u >> lg_us);
    const int64_t col = col0 + static_cast<int64_t>(u & us_mask) * (kPcThreads * VEC);
    live[u] = row < rows && col < inner;
    if (live[u]) held[u] = op.load4(row * inner + col);
  }
#pragma unroll
  for (int u = 0; u < kPcAccesses; ++u) {
    const int64_t row = row0 + (u >> lg_us);
    if (row >= rows) break;  // uniform
    int64_t c = c0 + (u >> lg_us);
    while (c >= C) c -= C;   // at most A - 1 rows past c0: uniform, a few scalar steps
    const typename Op::P p = op.params(c);
    const int64_t col = col0 + static_cast<int64_t>(u & us_mask) * (kPcThreads * VEC);
    if (live[u]) op.put4(row * inner + col, op.conv4(held[u], {p, p, p, p}));
  }
}

// Quotient and remainder of non-negative 32-bit values by a divisor whose fp32 reciprocal is
// at hand; exact for quotients below 2**20 (the estimate is off by one at most).
__device__ __forceinline__ void divmod_by(int a, int d, float inv_d, int& quo, int& rem) {
  quo = static_cast<int>(static_cast<float>(a) * inv_d);
  rem = a - quo * d;
  if (rem < 0) {
    --quo;
    rem += d;
  } else if (rem >= d) {
    ++quo;
    rem -= d;
  }
}

// pc_flat_kernel: rows that no 16-byte access divides (a weight of 5411 columns, 3 x 3 x 3
// taps) as one flat run.  A thread's group of four values begins in channel c and may run
// into c + 1; one 64-bit division per block, float-reciprocal ones per group, and each
// thread's own channel parameters from the caches while its values are on their way.
// Bound by memory like the row kernel: fp32 [8328, 5411] axis 0 (quantize) runs at the
// row kernel's rate, where the 4-byte accesses it replaces reached half of it.
constexpr int kPcFlatGroups = 4;  // groups of four values per thread
constexpr int64_t kPcFlatSpan = kPcThreads * kPcFlatGroups * 4;
constexpr int64_t kPcFlatMaxExtent = int64_t{1} << 30;  // inner and C within 32-bit arithmetic
template <class Op, bool VEC>
__global__ __launch_bounds__(kPcThreads) void pc_flat_kernel(Op op, int64_t n, int32_t C, int32_t inner, float inv_c,
                                                           float inv_inner, PcCheck check) {
  const int64_t block = pc_block(op, C, check);
  if (block < 0) return;
  const int64_t start = block * kPcFlatSpan;
  typename Op::In4 held[kPcFlatGroups];
  const int at0 = static_cast<int>(threadIdx.x) * 4;
#pragma unroll
  for (int u = 0; u < kPcFlatGroups; ++u) {
    const int64_t i = start + u * (kPcThreads * 4) + at0;
    if (VEC && i + 4 <= n) held[u] = op.load4(i);
  }
  const int64_t row0 = start / inner;
  const int rem0 = static_cast<int>(start - row0 * inner);
  const int c0 = static_cast<int>(row0 % C);
#pragma unroll
  for (int u = 0; u < kPcFlatGroups; ++u) {
    const int local = u * (kPcThreads * 4) + at0;
    const int64_t i = start + local;
    if (i >= n) break;
    int row, rem, wraps, c;
    divmod_by(rem0 + local, inner, inv_inner, row, rem);
    divmod_by(c0 + row, C, inv_c, wraps, c);
    const int first = inner - rem;  // values of this group that belong to channel c
    const typename Op::P a = op.params(c);
    typename Op::P b = a;
    if (first < 4) b = op.params(c + 1 == C ? 0 : c + 1);
    if (VEC && i + 4 <= n) {
      op.put4(i, op.conv4(held[u], {a, first > 1 ? a : b, first > 2 ? a : b, first > 3 ? a : b}));
    } else {
      for (int j = 0; j < 4 && i + j < n; ++j) op.put1(i + j, op.load1(i + j), j < first ? a : b);
    }
  }
}

// pc_cols_kernel: `rows` x C values whose channel is the column.  A block takes the columns
// [col0, col0 + width) of kPcColsRows runs of rows; its threads stand on `lanes` = width / VEC column
// groups x 256 / lanes rows, so every thread keeps its columns and their parameters.
constexpr int kPcColsThreads = 256;
constexpr int kPcColsSteps = 8;  // rows per thread
template <class Op, int VEC>
__global__ __launch_bounds__(kPcColsThreads) void pc_cols_kernel(Op op, int64_t rows, int64_t C, int32_t lanes,
                                                               uint32_t col_blocks, PcCheck check) {
  const int64_t block = pc_block(op, C, check);
  if (block < 0) return;
  const uint32_t rb = static_cast<uint32_t>(block) / col_blocks, cb = static_cast<uint32_t>(block) - rb * col_blocks;
  const int per = kPcColsThreads / lanes;  // rows side by side
  const int mine = static_cast<int>(threadIdx.x) / lanes;
  const int64_t col = (static_cast<int64_t>(cb) * lanes + (static_cast<int>(threadIdx.x) - mine * lanes)) * VEC;
  if (mine >= per || col >= C) return;
  const int64_t row0 = static_cast<int64_t>(rb) * (per * kPcColsSteps) + mine;
  std::conditional_t<VEC == 4, typename Op::In4, typename Op::In1> held[kPcColsSteps];
#pragma unroll
  for (int u = 0; u < kPcColsSteps; ++u) {
    const int64_t row = row0 + u * per;
    if (row < rows) {
      if constexpr (VEC == 4) held[u] = op.load4(row * C + col);
      else held[u] = op.load1(row * C + col);
    }
  }
  typename Op::P p[4];
#pragma unroll
  for (int j = 0; j < VEC; ++j) p[j] = op.params(col + j);
#pragma unroll
  for (int u = 0; u < kPcColsSteps; ++u) {
    const int64_t row = row0 + u * per;
    if (row < rows) {
      if constexpr (VEC == 4) op.put4(row * C + col, op.conv4(held[u], p));
      else op.put1(row * C + col, held[u], p[0]);
    }
  }
}

template <class Op>
__global__ __launch_bounds__(kThreads) void pc_element_kernel(Op op, int64_t n, int64_t C, int64_t inner, PcCheck check) {
  const int64_t block = pc_block(op, C, check);
  if (block < 0) return;
  const int64_t stride = (static_cast<int64_t>(gridDim.x) - (check.report != nullptr ? 1 : 0)) * kThreads;
  for (int64_t i = block * kThreads + threadIdx.x; i < n; i += stride)
    op.put1(i, op.load1(i), op.params((i / inner) % C));
}

inline unsigned grid_for(int64_t work_items, int64_t per_block, int64_t cap) {
  int64_t g = ceil_div(work_items, per_block);
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return static_cast<unsigned>(g);
}

// Codes that leave past the L2s, us without | with them, both directions: [11008, 4096] 69.3 | 67.1, [12288, 8192] 146.8 | 144.7,
// [12288, 12288] 217.9 | 215.1; [4096, 4096] level, [4096, 2048] 25.4 | 28.8 (as for the per-tensor quantizer above).
bool pc_through(int64_t n) { return n >= (int64_t{28} << 20); }

// `vec`: both pointers take 16-byte accesses of fp32 and 4-byte accesses of codes.
template <class Op>
int launch_per_channel(const Op& op, int64_t outer, int64_t C, int64_t inner, bool vec, const PcCheck& check,
                       hipStream_t s) {
  const int64_t n = outer * C * inner, extra = check.report != nullptr ? 1 : 0;
  if (n == 0) return TMQ_OK;
  if (inner == 1) {
    const bool v4 = vec && C % 4 == 0;
    const int64_t groups = v4 ? C / 4 : C;
    // as few column blocks as 256 threads allow, of equal width
    const int64_t col_blocks = ceil_div(groups, kPcColsThreads), lanes = ceil_div(groups, col_blocks);
    const int64_t blocks = ceil_div(outer, kPcColsThreads / lanes * kPcColsSteps) * col_blocks;
    if (blocks < 0x7fffffff) {
      const dim3 grid(static_cast<unsigned>(blocks + extra));
      if (v4)
        enqueue(pc_cols_kernel<Op, 4>, grid, dim3(kPcColsThreads), 0, s, op, outer, C, static_cast<int32_t>(lanes),
                static_cast<uint32_t>(col_blocks), check);
      else
        enqueue(pc_cols_kernel<Op, 1>, grid, dim3(kPcColsThreads), 0, s, op, outer, C, static_cast<int32_t>(lanes),
                static_cast<uint32_t>(col_blocks), check);
      return launch_status();
    }
  }
  if (vec && inner % 4 == 0 && inner >= kPcRowsMinInner) {
    constexpr int kPcAccesses = Op::kAccesses;
    const int64_t per_run = kPcThreads * 4;
    int lg_us = 0;
    while ((2 << lg_us) <= kPcAccesses && (per_run << lg_us) < inner) ++lg_us;
    const int64_t segs = ceil_div(inner, per_run << lg_us);
    const int64_t row_groups = ceil_div(outer * C, kPcAccesses >> lg_us);
    if (segs < 0x7fffffff && row_groups < 0x7fffffff / segs) {
      const auto rows = [&](const auto& stores) {
        enqueue(pc_rows_kernel<std::decay_t<decltype(stores)>>, dim3(static_cast<unsigned>(row_groups * segs + extra)),
                dim3(kPcThreads), 0, s, stores, outer * C, C, inner, lg_us, static_cast<uint32_t>(segs), check);
        return launch_status();
      };
      if constexpr (std::is_same_v<typename Op::Out4, uint32_t>) {  // a quantizer
        if (pc_through(n)) return rows(PcThrough<Op>(op));
      }
      return rows(op);
    }
  }
  if (inner >= 4 && inner <= kPcFlatMaxExtent && C <= kPcFlatMaxExtent && ceil_div(n, kPcFlatSpan) < 0x7fffffff) {
    const dim3 grid(static_cast<unsigned>(ceil_div(n, kPcFlatSpan) + extra));
    const int32_t c32 = static_cast<int32_t>(C), inner32 = static_cast<int32_t>(inner);
    const float inv_c = 1.0f / static_cast<float>(C), inv_inner = 1.0f / static_cast<float>(inner);
    if (vec)
      enqueue(pc_flat_kernel<Op, true>, grid, dim3(kPcThreads), 0, s, op, n, c32, inner32, inv_c, inv_inner, check);
    else
      enqueue(pc_flat_kernel<Op, false>, grid, dim3(kPcThreads), 0, s, op, n, c32, inner32, inv_c, inv_inner, check);
    return launch_status();
  }
  const unsigned g = grid_for(n, kThreads, 1 << 20);
  enqueue(pc_element_kernel<Op>, dim3(g + static_cast<unsigned>(extra)), dim3(kThreads), 0, s, op, n, C, inner, check);
  return launch_status();
}

// Codes that leave past the L2s (st4_through), us without | with them, quantize and dequantize: 32 Mi values 51.6 | 49.7, 48 Mi
// 74.6 | 73.2, 64 Mi 97.5 | 96.8, 128 Mi 191.0 | 191.2.  Fewer than the L2s hold stay in them for a dequantizer, whose blocks
// read what the same XCD wrote (24 Mi 36.8 | 38.1, 8 Mi 13.7 | 15.0).
bool quantize_through(int64_t n) { return n >= (int64_t{28} << 20) && n < (int64_t{96} << 20); }

template <bool SIGNED, bool FUSED>
int quantize_launch_as(const float* x, void* q, int64_t n, QParamsArg qp, hipStream_t s) {
  uint8_t* qb = static_cast<uint8_t*>(q);
  if (aligned(x, 16) && aligned(q, 4)) {
    const int64_t n4 = n / 4;
    const int64_t blocks = n4 == 0 ? 1 : ceil_div(n4, kQThreads * kUnrollQD);
    if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
    if (n > kStreamOutCodes)
      enqueue(quantize_vec_kernel<SIGNED, FUSED, kQStream>, dim3(blocks), dim3(kQThreads), 0, s,
              reinterpret_cast<const v4f*>(x), reinterpret_cast<uint32_t*>(q), n4, x, qb, n, qp);
    else if (quantize_through(n))
      enqueue(quantize_vec_kernel<SIGNED, FUSED, kQThrough>, dim3(blocks), dim3(kQThreads), 0, s,
              reinterpret_cast<const v4f*>(x), reinterpret_cast<uint32_t*>(q), n4, x, qb, n, qp);
    else
      enqueue(quantize_vec_kernel<SIGNED, FUSED>, dim3(blocks), dim3(kQThreads), 0, s,
              reinterpret_cast<const v4f*>(x), reinterpret_cast<uint32_t*>(q), n4, x, qb, n, qp);
  } else {
    const unsigned g = grid_for(n, kThreads, 65536);
    enqueue(quantize_scalar_kernel<SIGNED, FUSED>, dim3(g), dim3(kThreads), 0, s, x, qb, n, qp);
  }
  return launch_status();
}

int quantize_launch(const float* x, void* q, int64_t n, QParamsArg qp, int q_signed, hipStream_t s,
                    bool fused = false) {
  if (n == 0) return TMQ_OK;
  if (fused)
    return q_signed ? quantize_launch_as<true, true>(x, q, n, qp, s) : quantize_launch_as<false, true>(x, q, n, qp, s);
  return q_signed ? quantize_launch_as<true, false>(x, q, n, qp, s) : quantize_launch_as<false, false>(x, q, n, qp, s);
}

bool zp_in_range(int64_t zp, int q_signed) {
  return q_signed ? (zp >= -128 && zp <= 127) : (zp >= 0 && zp <= 255);
}

}  // namespace
}  // namespace tmq

using namespace tmq;

TMQ_EXPORT int tmq_quantize_per_tensor(const float* x, void* q, int64_t n, double scale,
                                       int64_t zero_point, int q_signed, tmq_stream_t stream) {
  if (n < 0 || (n > 0 && (x == nullptr || q == nullptr))) return TMQ_ERR_INVALID_ARGUMENT;
  if (!zp_in_range(zero_point, q_signed)) return TMQ_ERR_INVALID_ARGUMENT;
  QParamsArg qp;
  qp.inv = 1.0f / static_cast<float>(scale);
  qp.zp_f = static_cast<float>(zero_point);
  qp.dev = nullptr;
  return quantize_launch(x, q, n, qp, q_signed, as_stream(stream));
}

TMQ_EXPORT int tmq_quantize_per_tensor_dev(const float* x, void* q, int64_t n,
                                           const tmq_qparams* qparams, int q_signed,
                                           tmq_stream_t stream) {
  if (n < 0 || qparams == nullptr || (n > 0 && (x == nullptr || q == nullptr)))
    return TMQ_ERR_INVALID_ARGUMENT;
  QParamsArg qp;
  qp.inv = 0.f;
  qp.zp_f = 0.f;
  qp.dev = qparams;
  return quantize_launch(x, q, n, qp, q_signed, as_stream(stream));
}

TMQ_EXPORT int tmq_dequantize_per_tensor(const void* q, float* r, int64_t n, double scale,
                                         int64_t zero_point, int q_signed, tmq_stream_t stream) {
  if (n < 0 || (n > 0 && (r == nullptr || q == nullptr))) return TMQ_ERR_INVALID_ARGUMENT;
  if (!zp_in_range(zero_point, q_signed)) return TMQ_ERR_INVALID_ARGUMENT;
  if (n == 0) return TMQ_OK;
  hipStream_t s = as_stream(stream);
  const float scale_f = static_cast<float>(scale);
  const int zp = static_cast<int>(zero_point);
  const uint8_t* qb = static_cast<const uint8_t*>(q);
  if (aligned(r, 16) && aligned(q, 4)) {
    const int64_t n4 = n / 4;
    const int64_t blocks = n4 == 0 ? 1 : ceil_div(n4, kDqThreads * kUnrollQD);
    if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
    auto* q4 = reinterpret_cast<const uint32_t*>(q);
    auto* r4 = reinterpret_cast<v4f*>(r);
    if (q_signed)
      enqueue(dequantize_vec_kernel<true>, dim3(blocks), dim3(kDqThreads), 0, s, q4, r4, n4, qb, r, n, scale_f, zp);
    else
      enqueue(dequantize_vec_kernel<false>, dim3(blocks), dim3(kDqThreads), 0, s, q4, r4, n4, qb, r, n, scale_f, zp);
  } else {
    const unsigned g = grid_for(n, kThreads, 65536);
    if (q_signed)
      enqueue(dequantize_scalar_kernel<true>, dim3(g), dim3(kThreads), 0, s, qb, r, n, scale_f, zp);
    else
      enqueue(dequantize_scalar_kernel<false>, dim3(g), dim3(kThreads), 0, s, qb, r, n, scale_f, zp);
  }
  return launch_status();
}

TMQ_EXPORT size_t tmq_minmax_workspace_bytes(int64_t n) {
  (void)n;
  return static_cast<size_t>(kMinMaxMaxBlocks) * 2 * sizeof(float);
}

TMQ_EXPORT int tmq_minmax(const float* x, int64_t n, float* minmax, void* workspace,
                          size_t workspace_bytes, tmq_stream_t stream) {
  if (n < 0 || minmax == nullptr || (n > 0 && x == nullptr)) return TMQ_ERR_INVALID_ARGUMENT;
  if (workspace == nullptr || workspace_bytes < tmq_minmax_workspace_bytes(n) ||
      !aligned(workspace, 4))
    return TMQ_ERR_WORKSPACE;
  if (!aligned(x, 4)) return TMQ_ERR_ALIGNMENT;
  hipStream_t s = as_stream(stream);
  float* partials = static_cast<float*>(workspace);
  // elements before the first 16-byte boundary are handled one by one
  int64_t head = 0;
  if (n > 0) {
    const uintptr_t mis = reinterpret_cast<uintptr_t>(x) & 15u;
    head = mis == 0 ? 0 : static_cast<int64_t>((16 - mis) / 4);
    if (head > n) head = n;
  }
  const int64_t n4 = (n - head) / 4;
  const unsigned g = grid_for(n4, kThreads * kUnroll, kMinMaxMaxBlocks);
  enqueue(minmax_partial_kernel<false>, dim3(g), dim3(kThreads), 0, s,
          reinterpret_cast<const v4f*>(x + head), n4, x, head, n, partials, RangeReport{nullptr, 0, 0});
  if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  enqueue(minmax_final_kernel, dim3(1), dim3(kThreads), 0, s, partials, static_cast<int>(g), minmax);
  return launch_status();
}

TMQ_EXPORT int tmq_choose_qparams_dev(const float* minmax, int q_signed, int reduce_range,
                                      tmq_qparams* qparams, tmq_stream_t stream) {
  if (minmax == nullptr || qparams == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  enqueue(choose_qparams_kernel, dim3(1), dim3(kWave), 0, as_stream(stream),
          minmax, q_signed ? -128 : 0, q_signed ? 127 : 255, reduce_range, qparams);
  return launch_status();
}

namespace tmq {
namespace {

// ---------------------------------------------------------------------------
// Dynamic quantization in one launch whose blocks exchange their ranges (quantize_held.h): where it is taken and how.
// ---------------------------------------------------------------------------
// Above 32 Ki values; up to there dynamic_quantize_repeat_kernel (us, that | this: 16 Ki 3.5 | 3.3, 32 Ki 3.6 | 3.7, 64 Ki
// 4.8 | 4.0, 96 Ki 5.8 | 3.9).  Up to 64 Mi values; beyond, range and codes stream past the caches in three launches (64 Mi
// 94 | 87, 256 Mi 372 | 478: one block per CU has too little on its way for what it does not hold).
constexpr int64_t kHeldAbove = 32768, kHeldUpTo = int64_t{1} << 26;

struct HeldCall {
  const float* x;
  void* q;
  int64_t M, K, pitch;  // pitch == K: dense, M * K values
  int q_signed;
  bool fused;
  int reduce_range;
  tmq_qparams* qparams;
  void* workspace;
  size_t workspace_bytes;
};
// What the kernel needs of a call, whatever its size.
bool held_runs(const HeldCall& c, hipStream_t s) {
  const bool rows = c.pitch != c.K;
  if (c.fused && c.q_signed) return false;
  if (!aligned(c.q, 4) || !aligned(c.x, rows ? 4 : 16) || (rows && (!c.fused || c.K < 4 || c.M * (c.pitch / 4) > (1 << 30)))) return false;
  if (c.M * c.K < 4 || c.M * c.K > kHeldUpTo) return false;
  if (c.workspace == nullptr || c.workspace_bytes < kHeldBlocks * sizeof(v4u) || !aligned(c.workspace, 16)) return false;
  return cu_count() > 0 && !replayed(s);
}
template <bool FUSED, bool ROWS>
auto held_kernel(int held) {
  switch (held) {
    case 1: return dynamic_quantize_held_kernel<FUSED, ROWS, 1>;
    case 2: return dynamic_quantize_held_kernel<FUSED, ROWS, 2>;
    case 3: return dynamic_quantize_held_kernel<FUSED, ROWS, 3>;
    case 4: return dynamic_quantize_held_kernel<FUSED, ROWS, 4>;
    case 6: return dynamic_quantize_held_kernel<FUSED, ROWS, 6>;
    case 8: return dynamic_quantize_held_kernel<FUSED, ROWS, 8>;
    case 12: return dynamic_quantize_held_kernel<FUSED, ROWS, 12>;
    case 16: return dynamic_quantize_held_kernel<FUSED, ROWS, 16>;
    case 24: return dynamic_quantize_held_kernel<FUSED, ROWS, 24>;
    default: return dynamic_quantize_held_kernel<FUSED, ROWS, kHeldMost>;
  }
}
// The host takes the range of up to TMQ_HOST_PARTS_UP_TO values in parts, from as many blocks as it has words for: each
// tells it its own, 1.5 us before any block knows all of them (with dequantize, against range pass and quantizer in two
// launches: 874 x 2752 values 19.5 -> 16.4 us, 128 x 1024 level at 13.9, where the host's own work is the time).
// polls: negative for as many as kRangePolls says.
int launch_held(const HeldCall& c, int most_blocks, int polls, const RangeReport& report, uint64_t* parts, int32_t* parts_count,
                hipStream_t s) {
  const bool rows = c.pitch != c.K;
  const int64_t n = c.M * c.K, total = rows ? c.M * (c.pitch / 4) : n / 4;
  int64_t blocks = ceil_div(total, kHeldThreads);
  blocks = std::min({blocks, int64_t{most_blocks}, int64_t{kHeldBlocks}, int64_t{cu_count()}});
  const int64_t per_thread = ceil_div(total, blocks * kHeldThreads);
  int held = kHeldMost;
  for (const int h : {24, 16, 12, 8, 6, 4, 3, 2, 1})
    if (h >= per_thread) held = h;
  const int32_t more = static_cast<int32_t>(per_thread > held ? per_thread - held : 0);
  const auto kernel = rows ? held_kernel<true, true>(held) : c.fused ? held_kernel<true, false>(held) : held_kernel<false, false>(held);
  const RangeWords range{static_cast<v4u*>(c.workspace), next_range_tag(), polls >= 0 ? polls : more > 0 ? 2 * kRangePolls : kRangePolls};
  if (parts != nullptr) *parts_count = static_cast<int32_t>(blocks);
  enqueue(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kHeldThreads), 0, s, c.x, static_cast<uint32_t*>(c.q),
          static_cast<int32_t>(total), static_cast<int32_t>(rows ? c.K : 0), static_cast<int32_t>(rows ? c.pitch / 4 : 1),
          static_cast<int32_t>(rows ? 0 : n % 4), range, more, c.q_signed ? 0x80808080u : 0u, c.q_signed ? -128 : 0,
          c.q_signed ? 127 : 255, c.reduce_range, c.qparams, report, parts);
  return launch_status();
}

int quantize_dynamic(const float* x, void* q, int64_t n, int q_signed, int reduce_range, int rounding,
                     tmq_qparams* qparams, void* workspace, size_t workspace_bytes, RangeReport report,
                     tmq_stream_t stream, uint64_t* parts = nullptr, int32_t* parts_count = nullptr) {
  if (n < 0 || qparams == nullptr || (n > 0 && (x == nullptr || q == nullptr))) return TMQ_ERR_INVALID_ARGUMENT;
  if (rounding != TMQ_ROUND_PRODUCT && rounding != TMQ_ROUND_FUSED) return TMQ_ERR_INVALID_ARGUMENT;
  const bool fused = rounding == TMQ_ROUND_FUSED;
  if (!aligned(x, 4)) return TMQ_ERR_ALIGNMENT;
  hipStream_t s = as_stream(stream);
  const int qmin = q_signed ? -128 : 0, qmax = q_signed ? 127 : 255;
  const bool vec_ok = aligned(x, 16) && aligned(q, 4);
  const bool two_ok = workspace != nullptr && workspace_bytes >= tmq_minmax_workspace_bytes(n) && aligned(workspace, 8);
  const HeldCall held{x, q, 1, n, n, q_signed, fused, reduce_range, qparams, workspace, workspace_bytes};
  if (n > kHeldAbove && held_runs(held, s)) {
    const bool in_parts = parts != nullptr && n > TMQ_HOST_PARTS_ABOVE && n <= TMQ_HOST_PARTS_UP_TO;
    return launch_held(held, in_parts ? TMQ_HOST_PARTS : kHeldBlocks, -1, in_parts ? RangeReport{nullptr, 0, 0} : report,
                       in_parts ? parts : nullptr, parts_count, s);
  }
  if (n <= kDynRepeatMax) {
    const int32_t n32 = static_cast<int32_t>(n);
    // (nothing to quantize: one block still publishes the parameters)
    return launch_dynamic_repeat(q_signed != 0, fused, n > 0 ? ceil_div(n, 4) : 1, s, x, static_cast<uint8_t*>(q), n32, n32, 0,
                                 qmin, qmax, reduce_range, aligned(q, 4), qparams, report);
  }
  if (workspace == nullptr || workspace_bytes < tmq_minmax_workspace_bytes(n) ||
      !aligned(workspace, report.to != nullptr ? 8 : 4))
    return TMQ_ERR_WORKSPACE;
  float* partials = static_cast<float*>(workspace);
  const RangeReport none{nullptr, 0, 0};
  if (n <= kDynKeepMax && vec_ok && two_ok) {
    // Inputs that fit the last-level cache with room to spare (where the launches, not the
    // bytes, are what counts): two launches -- partial ranges, read with ordinary loads so
    // that the second pass finds the input cached, then the quantizer whose blocks finish
    // the reduction themselves.
    const RangeReport early = n <= kDynEarlyMax ? report : none, late = n <= kDynEarlyMax ? none : report;
    const int64_t n4 = n / 4;
    const unsigned g = grid_for(n4, kThreads * kUnroll, kDynPartials);
    const v4f* x4 = reinterpret_cast<const v4f*>(x);
    enqueue(minmax_partial_kernel<true>, dim3(g), dim3(kThreads), 0, s, x4, n4, x, 0, n, partials, early);
    if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
    const dim3 grid(grid_for(n4, kThreads * kUnrollQD, kDynQBlocks)), block(kThreads);
    uint32_t* q4 = static_cast<uint32_t*>(q);
    uint8_t* qb = static_cast<uint8_t*>(q);
    const int cnt = static_cast<int>(g);
    if (q_signed && fused)
      enqueue(quantize_after_minmax_kernel<true, true>, grid, block, 0, s,
              x4, q4, n4, x, qb, n, partials, cnt, qmin, qmax, reduce_range, qparams, late);
    else if (q_signed)
      enqueue(quantize_after_minmax_kernel<true, false>, grid, block, 0, s,
              x4, q4, n4, x, qb, n, partials, cnt, qmin, qmax, reduce_range, qparams, late);
    else if (fused)
      enqueue(quantize_after_minmax_kernel<false, true>, grid, block, 0, s,
              x4, q4, n4, x, qb, n, partials, cnt, qmin, qmax, reduce_range, qparams, late);
    else
      enqueue(quantize_after_minmax_kernel<false, false>, grid, block, 0, s,
              x4, q4, n4, x, qb, n, partials, cnt, qmin, qmax, reduce_range, qparams, late);
    return launch_status();
  }
  // larger inputs (streamed past the caches) and unaligned buffers: range, parameters and
  // codes in three launches
  const uintptr_t mis = reinterpret_cast<uintptr_t>(x) & 15u;
  int64_t head = mis == 0 ? 0 : static_cast<int64_t>((16 - mis) / 4);
  if (head > n) head = n;
  const int64_t n4 = (n - head) / 4;
  const unsigned g = grid_for(n4, kThreads * kUnroll, kMinMaxMaxBlocks);
  enqueue(minmax_partial_kernel<false>, dim3(g), dim3(kThreads), 0, s, reinterpret_cast<const v4f*>(x + head), n4, x, head,
          n, partials, none);
  if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  enqueue(minmax_final_choose_kernel, dim3(1), dim3(kThreads), 0, s, partials, static_cast<int>(g), qmin, qmax,
          reduce_range, qparams, report);
  if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  QParamsArg qp;
  qp.inv = 0.f;
  qp.zp_f = 0.f;
  qp.dev = qparams;
  return quantize_launch(x, q, n, qp, q_signed, s, fused);
}
}  // namespace
}  // namespace tmq

TMQ_EXPORT int tmq_quantize_per_tensor_dynamic_dev(const float* x, void* q, int64_t n, int q_signed,
                                                   int reduce_range, int rounding, tmq_qparams* qparams,
                                                   void* workspace, size_t workspace_bytes, tmq_stream_t stream) {
  return quantize_dynamic(x, q, n, q_signed, reduce_range, rounding, qparams, workspace, workspace_bytes,
                          RangeReport{nullptr, 0, 0}, stream);
}

TMQ_EXPORT int tmq_quantize_per_tensor_dynamic_report(const float* x, void* q, int64_t n, int q_signed,
                                                      int reduce_range, int rounding, tmq_qparams* qparams,
                                                      void* workspace, size_t workspace_bytes,
                                                      tmq_host_report* report, uint32_t ticket, uint32_t slot,
                                                      tmq_stream_t stream) {
  if (report == nullptr || n <= 0 || slot >= TMQ_HOST_REPORTS) return TMQ_ERR_INVALID_ARGUMENT;
  return quantize_dynamic(x, q, n, q_signed, reduce_range, rounding, qparams, workspace, workspace_bytes,
                          RangeReport{report, ticket, slot}, stream);
}

TMQ_EXPORT int tmq_quantize_per_tensor_dynamic_parts(const float* x, void* q, int64_t n, int q_signed,
                                                     int reduce_range, int rounding, tmq_qparams* qparams,
                                                     void* workspace, size_t workspace_bytes,
                                                     tmq_host_report* report, uint32_t ticket, uint32_t slot,
                                                     uint64_t* parts, int32_t* count, tmq_stream_t stream) {
  if (report == nullptr || n <= 0 || slot >= TMQ_HOST_REPORTS || parts == nullptr || count == nullptr || !aligned(parts, 8))
    return TMQ_ERR_INVALID_ARGUMENT;
  *count = 0;
  return quantize_dynamic(x, q, n, q_signed, reduce_range, rounding, qparams, workspace, workspace_bytes,
                          RangeReport{report, ticket, slot}, stream, parts, count);
}

TMQ_EXPORT int tmq_quantize_rows_dynamic_dev(const float* x, void* q, int64_t M, int64_t K, int64_t pitch, int q_signed,
                                             int reduce_range, int rounding, tmq_qparams* qparams, void* workspace,
                                             size_t workspace_bytes, tmq_stream_t stream) {
  if (M < 1 || K < 1 || K > 0x7fffff00 || pitch % 16 != 0 || pitch < K || x == nullptr || q == nullptr || qparams == nullptr)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (rounding != TMQ_ROUND_PRODUCT && rounding != TMQ_ROUND_FUSED) return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(x, 4) || !aligned(q, 4)) return TMQ_ERR_ALIGNMENT;
  if (workspace == nullptr || workspace_bytes < tmq_minmax_workspace_bytes(M * K) || !aligned(workspace, 8))
    return TMQ_ERR_WORKSPACE;
  hipStream_t s = as_stream(stream);
  const int qmin = q_signed ? -128 : 0, qmax = q_signed ? 127 : 255;
  const bool fused = rounding == TMQ_ROUND_FUSED;
  const int64_t n = M * K;
  const HeldCall held{x, q, M, K, pitch, q_signed, fused, reduce_range, qparams, workspace, workspace_bytes};
  if (n > kHeldAbove && held_runs(held, s))
    return launch_held(held, kHeldBlocks, -1, RangeReport{nullptr, 0, 0}, nullptr, nullptr, s);
  if (n <= kDynRepeatMax)
    return launch_dynamic_repeat(q_signed != 0, fused, M * (pitch / 4), s, x, static_cast<uint8_t*>(q), static_cast<int32_t>(n),
                                 static_cast<int32_t>(K), static_cast<int32_t>(pitch / 4), qmin, qmax, reduce_range, true,
                                 qparams, RangeReport{nullptr, 0, 0});
  float* partials = static_cast<float*>(workspace);
  const uintptr_t mis = reinterpret_cast<uintptr_t>(x) & 15u;
  int64_t head = mis == 0 ? 0 : static_cast<int64_t>((16 - mis) / 4);
  if (head > n) head = n;
  const int64_t n4 = (n - head) / 4;
  const int count = static_cast<int>(grid_for(n4, kThreads * kUnroll, kDynPartials));
  enqueue(minmax_partial_kernel<true>, dim3(count), dim3(kThreads), 0, s,
          reinterpret_cast<const v4f*>(x + head), n4, x, head, n,
          partials, RangeReport{nullptr, 0, 0});
  if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  const dim3 grid(grid_for(M * (pitch / 4), kThreads * 2, kDynQBlocks)), block(kThreads);
  auto go = [&](auto kernel) {
    enqueue(kernel, grid, block, 0, s, x, static_cast<uint32_t*>(q), M, static_cast<int32_t>(K), static_cast<int32_t>(pitch / 4),
            partials, count, qmin, qmax, reduce_range, qparams);
    return launch_status();
  };
  if (q_signed) return fused ? go(quantize_rows_after_minmax_kernel<true, true>) : go(quantize_rows_after_minmax_kernel<true, false>);
  return fused ? go(quantize_rows_after_minmax_kernel<false, true>) : go(quantize_rows_after_minmax_kernel<false, false>);
}

TMQ_EXPORT int tmq_quantize_dynamic_exchange(const float* x, void* q, int64_t M, int64_t K, int64_t pitch, int q_signed,
                                            int reduce_range, int rounding, tmq_qparams* qparams, void* workspace,
                                            size_t workspace_bytes, int blocks, int polls, tmq_stream_t stream) {
  if (M < 1 || K < 1 || K > 0x7fffff00 || pitch < K || (pitch != K && pitch % 16 != 0) || x == nullptr || q == nullptr ||
      qparams == nullptr || blocks < 1 || polls < 0 || M > (int64_t{1} << 40) / K)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (rounding != TMQ_ROUND_PRODUCT && rounding != TMQ_ROUND_FUSED) return TMQ_ERR_INVALID_ARGUMENT;
  const HeldCall held{x, q, M, K, pitch, q_signed, rounding == TMQ_ROUND_FUSED, reduce_range, qparams, workspace, workspace_bytes};
  if (!held_runs(held, as_stream(stream))) return TMQ_ERR_UNSUPPORTED;
  return launch_held(held, blocks, polls, RangeReport{nullptr, 0, 0}, nullptr, nullptr, as_stream(stream));
}

TMQ_EXPORT int tmq_choose_qparams_host(float min, float max, int q_signed, int reduce_range,
                                       double* scale, int32_t* zero_point) {
  if (scale == nullptr || zero_point == nullptr || !(min <= max)) return TMQ_ERR_INVALID_ARGUMENT;
  choose_qparams(min, max, q_signed ? -128 : 0, q_signed ? 127 : 255, reduce_range != 0, scale,
                 zero_point);
  return TMQ_OK;
}

TMQ_EXPORT int tmq_per_channel(const tmq_per_channel_desc* d, tmq_stream_t stream) {
  if (d == nullptr || d->outer < 0 || d->channels < 0 || d->inner < 0) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->outer == 0 || d->channels == 0 || d->inner == 0) return d->report == nullptr ? TMQ_OK : TMQ_ERR_INVALID_ARGUMENT;
  if (d->fp32 == nullptr || d->codes == nullptr || d->scales == nullptr || d->zero_points == nullptr)
    return TMQ_ERR_INVALID_ARGUMENT;
  hipStream_t s = as_stream(stream);
  const PcCheck check{d->report, d->ticket};
  auto* f = static_cast<float*>(d->fp32);
  auto* q = static_cast<uint8_t*>(d->codes);
  const bool vec = aligned(f, 16) && aligned(q, 4);
  auto go = [&](const auto& op) { return launch_per_channel(op, d->outer, d->channels, d->inner, vec, check, s); };
  if (d->float_qparams) {
    auto* sc = static_cast<const float*>(d->scales);
    auto* zp = static_cast<const float*>(d->zero_points);
    if (d->dequantize) return d->q_signed ? go(PcfDequantize<true>{q, f, sc, zp}) : go(PcfDequantize<false>{q, f, sc, zp});
    return d->q_signed ? go(PcfQuantize<true>{f, q, sc, zp}) : go(PcfQuantize<false>{f, q, sc, zp});
  }
  auto* sc = static_cast<const double*>(d->scales);
  auto* zp = static_cast<const int64_t*>(d->zero_points);
  if (d->dequantize) return d->q_signed ? go(PcDequantize<true>{q, f, sc, zp}) : go(PcDequantize<false>{q, f, sc, zp});
  return d->q_signed ? go(PcQuantize<true>{f, q, sc, zp}) : go(PcQuantize<false>{f, q, sc, zp});
}

namespace {
int per_channel(int dequantize, int float_qparams, const void* fp32, const void* codes, int64_t outer, int64_t channels,
                int64_t inner, const void* scales, const void* zero_points, int q_signed, tmq_stream_t stream) {
  tmq_per_channel_desc d{};
  d.dequantize = dequantize;
  d.float_qparams = float_qparams;
  d.q_signed = q_signed;
  d.fp32 = const_cast<void*>(fp32);
  d.codes = const_cast<void*>(codes);
  d.outer = outer;
  d.channels = channels;
  d.inner = inner;
  d.scales = scales;
  d.zero_points = zero_points;
  return tmq_per_channel(&d, stream);
}
}  // namespace

TMQ_EXPORT int tmq_quantize_per_channel(const float* x, void* q, int64_t outer, int64_t channels,
                                        int64_t inner, const double* scales,
                                        const int64_t* zero_points, int q_signed,
                                        tmq_stream_t stream) {
  return per_channel(0, 0, x, q, outer, channels, inner, scales, zero_points, q_signed, stream);
}

TMQ_EXPORT int tmq_dequantize_per_channel(const void* q, float* r, int64_t outer, int64_t channels,
                                          int64_t inner, const double* scales,
                                          const int64_t* zero_points, int q_signed,
                                          tmq_stream_t stream) {
  return per_channel(1, 0, r, q, outer, channels, inner, scales, zero_points, q_signed, stream);
}

TMQ_EXPORT int tmq_quantize_per_channel_float_qparams(const float* x, void* q, int64_t outer,
                                                      int64_t channels, int64_t inner,
                                                      const float* scales, const float* zero_points,
                                                      int q_signed, tmq_stream_t stream) {
  return per_channel(0, 1, x, q, outer, channels, inner, scales, zero_points, q_signed, stream);
}

TMQ_EXPORT int tmq_dequantize_per_channel_float_qparams(const void* q, float* r, int64_t outer,
                                                        int64_t channels, int64_t inner,
                                                        const float* scales, const float* zero_points,
                                                        int q_signed, tmq_stream_t stream) {
  return per_channel(1, 1, r, q, outer, channels, inner, scales, zero_points, q_signed, stream);
}

TMQ_EXPORT const char* tmq_status_string(int status) {
  switch (status) {
    case TMQ_OK: return "ok";
    case TMQ_ERR_INVALID_ARGUMENT: return "invalid argument";
    case TMQ_ERR_UNSUPPORTED: return "unsupported configuration";
    case TMQ_ERR_WORKSPACE: return "workspace missing or too small";
    case TMQ_ERR_LAUNCH: return "HIP launch failed";
    case TMQ_ERR_ALIGNMENT: return "pointer or leading dimension not aligned";
    default: return "unknown status";
  }
}

TMQ_EXPORT int tmq_version(void) { return TMQ_VERSION; }
