// Pieces of a dynamic quantization inside a block (device code for gfx950 only): minimum and maximum across a wave, float rows
// held in registers between their range and their codes.
#pragma once

#include "common.h"
#include "qparams.h"

namespace tmq {
namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_float(float v) {  // (lanes without a source keep their own value)
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ void minmax_step(float& mn, float& mx) {
  mn = fminf(mn, dpp_float<CTRL>(mn));
  mx = fmaxf(mx, dpp_float<CTRL>(mx));
}
// Minimum and maximum of each 16 lanes in the last of them (row_shr 1, 2, 4, 8) ...
__device__ __forceinline__ void row_minmax(float& mn, float& mx) {
  minmax_step<0x111>(mn, mx);
  minmax_step<0x112>(mn, mx);
  minmax_step<0x114>(mn, mx);
  minmax_step<0x118>(mn, mx);
}
// ... and of the wave in its last lane (row_bcast 15, 31).
__device__ __forceinline__ void wave_minmax_last(float& mn, float& mx) {
  row_minmax(mn, mx);
  minmax_step<0x142>(mn, mx);
  minmax_step<0x143>(mn, mx);
}
__device__ __forceinline__ float lane_float(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ void take_four(const v4f& v, float& mn, float& mx) {
  mn = fminf(fminf(mn, v.x), fminf(v.y, fminf(v.z, v.w)));
  mx = fmaxf(fmaxf(mx, v.x), fmaxf(v.y, fmaxf(v.z, v.w)));
}

// Four unsigned codes, product and zero point rounded once, as PyTorch's CPU quantized::linear_dynamic quantizes while it
// packs: v_cvt_pk_u8_f32 rounds to nearest even and saturates to [0, 255] (NaN -> 0).
__device__ __forceinline__ uint32_t fused_codes(const v4f& v, float inv, float zp_f) {
  uint32_t packed = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(v[j], inv, zp_f), j, packed);
  return packed;
}

// M rows of K >= 4 float values (4-byte aligned), all of them in a block's registers: thread t has groups t, t + THREADS, ... of
// four values, at most HELD, counted along the rows; a row's last group begins where its last four values do.  One division
// per thread and none per group (linear_resident.h has what that was worth).
struct __attribute__((packed, aligned(4))) FourFloats {
  v4f v;
};
template <int HELD, int THREADS>
struct HeldRows {
  v4f held[HELD];
  int K, k4, row0, c40, step_row, step_c4, M;

  __device__ __forceinline__ void next(int& row, int& c4) const {
    row += step_row;
    c4 += step_c4;
    if (c4 >= k4) {
      c4 -= k4;
      ++row;
    }
  }
  __device__ __forceinline__ void load(const float* __restrict__ x, int64_t ldx, int rows, int K_, int t) {
    M = rows;
    K = K_;
    k4 = (K + 3) >> 2;
    step_row = __builtin_amdgcn_readfirstlane(THREADS / k4);
    step_c4 = THREADS - step_row * k4;
    row0 = t / k4;
    c40 = t - row0 * k4;
    int row = row0, c4 = c40;
#pragma unroll
    for (int u = 0; u < HELD; ++u) {  // (unconditional loads keep the load counter exact; groups past the last: of row 0)
      const int c = 4 * c4 + 4 <= K ? 4 * c4 : K - 4;
      held[u] = reinterpret_cast<const FourFloats*>(x + (row < M ? row : 0) * ldx + c)->v;
      next(row, c4);
    }
  }
  __device__ __forceinline__ void range(float& mn, float& mx) const {
#pragma unroll
    for (int u = 0; u < HELD; ++u) take_four(held[u], mn, mx);
  }
  // put(row, c4, codes): values 4 c4 ... 4 c4 + 3 of a row; codes behind its end are those of other values of the row.
  template <class Put>
  __device__ __forceinline__ void codes(float inv, float zp_f, Put&& put) const {
    int row = row0, c4 = c40;
    asm volatile("" : "+v"(row), "+v"(c4));  // (walked again, not kept in 2 HELD registers since the loads)
#pragma unroll
    for (int u = 0; u < HELD; ++u) {
      uint32_t q = fused_codes(held[u], inv, zp_f);
      const int past = 4 * c4 + 4 - K;  // a last group's codes move down by the values it shares with the one before
      if (past > 0) q >>= 8 * past;
      if (row < M) put(row, c4, q);
      next(row, c4);
    }
  }
};

// The block's range and what follows from it, in every thread: each wave's minimum and maximum come in, `shared` is 2 W + 3
// floats of LDS; two barriers.
template <int W, class Barrier>
__device__ __forceinline__ void block_qparams(float mn, float mx, float* shared, int t, bool reduce_range, Barrier&& barrier,
                                              float& scale, float& inv, float& zp_f) {
  static_assert(W <= 16 && 16 % W == 0);
  wave_minmax_last(mn, mx);
  if (t % kWave == kWave - 1) {
    shared[t / kWave] = mn;
    shared[W + t / kWave] = mx;
  }
  barrier();
  if (t < kWave) {
    mn = shared[t % W];
    mx = shared[W + t % W];
    row_minmax(mn, mx);
    double s;
    int32_t z;
    choose_qparams(lane_float(mn, 15), lane_float(mx, 15), 0, 255, reduce_range, &s, &z);
    if (t == 0) {
      const float scf = static_cast<float>(s);
      shared[2 * W] = scf;
      shared[2 * W + 1] = 1.0f / scf;  // IEEE division, as the separate quantize kernels
      shared[2 * W + 2] = static_cast<float>(z);
    }
  }
  barrier();
  scale = shared[2 * W];
  inv = shared[2 * W + 1];
  zp_f = shared[2 * W + 2];
}

}  // namespace
}  // namespace tmq
