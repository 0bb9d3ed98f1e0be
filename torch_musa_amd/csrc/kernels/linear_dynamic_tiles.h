// quantized::linear_dynamic for more than 16 rows in one launch (gfx950): one round of tiles of 32 rows x 32 or 64 channels whose
// blocks read their float rows, tell each other the rows' ranges, and multiply the codes they make of them.
//
// What bounds such a call in two launches is the launches: 8 us for a product of any size, of which the codes' kernel and the
// product's own chain (start, first bytes, last barrier) are half each, and the host queues two.  Us, the launches before | this
// one: 441 x 213 -> 64 10.3 | 5.0, 60 x 128 -> 256 7.5 | 4.9, 412 x 208 -> 1216 10.1 | 5.3, 2456 x 451 -> 150 12.9 | 5.9, 68 x 1024 ->
// 2944 9.9 | 6.5, 347 x 1775 -> 424 12.3 | 9.0, 22 x 64 -> 176 (no exchange) 7.3 | 4.2; 56 drawn shapes 0.62 of the time, none slower.
// Here the product's requests -- the
// wave's float rows, then its weights -- leave before anything is known about the range, and the exchange (range_exchange.h, about
// 1.5 us) passes under the weights.  The rows come in as floats once for every tile of channels, which is what the split costs: 4 K
// bytes a row from the L2s where the codes are K, so K ends at 2048 and the XCDs take runs of tiles that share the larger operand.
//
// The eight waves of a block split K into shares of S values: a wave holds its share of the block's 32 rows in registers (S / 2
// of them, 1 KB a request) from the range to the codes, puts the codes into its own LDS in wloop's layout (gemm_i8_wloop.h),
// multiplies them with its share of the weights, also in registers by then, and the partial tiles meet behind one barrier.
#pragma once

#include "dynamic_rows.h"
#include "gemm_i8_wloop.h"
#include "range_exchange.h"

namespace tmq {

constexpr int kDynTileWaves = 8, kDynTileThreads = kDynTileWaves * kWave;

// Block -> tile: the operand that one XCD's run of tiles shares is the rows (by_rows) or the channels.
struct DynTileOrder {
  uint32_t tiles_m, tiles_n, reciprocal;  // 2^32 / (by_rows ? tiles_n : tiles_m), rounded up; 0 for a divisor of 1
  int32_t by_rows;
};

template <int CT, int S>
__global__ __launch_bounds__(kDynTileThreads, S <= 64 ? 4 : 2) void linear_dynamic_tiles_kernel(GemmArgs a, const float* __restrict__ x, int64_t ldx,
                                                                                  int reduce_range, RangeWords range,
                                                                                  DynTileOrder order) {
  constexpr int BM = 32, BN = 32 * CT, WAVES = kDynTileWaves;
  constexpr int kLanes = S / 4, kRows = kWave / kLanes, R = BM / kRows;  // lanes a row, rows a request, requests
  constexpr int kSteps = S / 32, kSlots = S / 16;
  constexpr int kRedPitch = BN * 4 + 16;
  constexpr int kWaveLds = BM * S > BM * kRedPitch ? BM * S : BM * kRedPitch;  // the wave's codes, then its partial tile
  __shared__ __attribute__((aligned(16))) uint8_t sX[WAVES][kWaveLds];
  __shared__ __attribute__((aligned(16))) int s_raw[3][kWave];  // colsum, weight scale, bias as fetched
  __shared__ float s_range[2 * WAVES], s_scale, s_inv, s_zp;
  __shared__ int s_missing;

  const int t = threadIdx.x, lane = t % kWave;
  const int wave_u = __builtin_amdgcn_readfirstlane(t / kWave);
  const int li = lane & 31, half = lane >> 5;
  const int K = static_cast<int>(a.K);
  const uint32_t all = gridDim.x, xcd = blockIdx.x % 8;
  const uint32_t tile = xcd * (all / 8) + (xcd < all % 8 ? xcd : all % 8) + blockIdx.x / 8;
  const uint32_t minor = order.by_rows != 0 ? order.tiles_n : order.tiles_m;
  const uint32_t major_at = order.reciprocal != 0 ? __umulhi(tile, order.reciprocal) : tile, minor_at = tile - major_at * minor;
  const int tile_m = static_cast<int>(order.by_rows != 0 ? major_at : minor_at);
  const int tile_n = static_cast<int>(order.by_rows != 0 ? minor_at : major_at);
  const int tiles_m = static_cast<int>(order.tiles_m);
  const int64_t m0 = static_cast<int64_t>(tile_m) * BM, n0 = static_cast<int64_t>(tile_n) * BN;

  // ---- requests: the wave's share of the rows (groups of four values; behind K: a row's last four again) ...
  const int c = wave_u * S + 4 * (lane % kLanes);
  v4f held[R];
  {
    const float* const xtile = x + m0 * ldx + (c + 4 <= K ? c : K - 4);
    const int64_t m_last = a.M - 1 - m0;     // rows past M: the last one again
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = i * kRows + lane / kLanes;
      held[i] = reinterpret_cast<const FourFloats*>(xtile + (r < m_last ? r : m_last) * ldx)->v;
    }
  }
  // ... and of the weights, and the tile's constants
  v4i w[CT][kSteps];
  {
    const int kc_last = static_cast<int>(a.w_kchunks) - 1;
    const int64_t nb_last = ceil_div(a.N, 16) - 1 - n0 / 16;  // 16-row blocks past N: clamped, never stored
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int64_t rb0 = 2 * ct + ((lane >> 4) & 1);
      const uint8_t* const wlane = a.w_packed + (n0 / 16 + (rb0 < nb_last ? rb0 : nb_last)) * a.w_kchunks * 256 + (lane & 15) * 16;
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        const int kc = wave_u * kSlots + 2 * j + half;
        w[ct][j] = ld16(wlane + static_cast<int64_t>(kc < kc_last ? kc : kc_last) * 256);
      }
    }
  }
  const int64_t n_raw = n0 + t % BN < a.N ? n0 + t % BN : a.N - 1;
  const int colsum = a.colsum[n_raw];
  const int scale = __float_as_int(a.w_scales[n_raw * a.w_scale_stride]);
  const int bias = __float_as_int((a.bias != nullptr ? a.bias : a.w_scales)[a.bias != nullptr ? n_raw : 0]);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the range of the block's rows, then of all of them
  float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < R; ++i) take_four(held[i], mn, mx);
  block_range<WAVES>(mn, mx, s_range, t);
  if (tiles_m > 1 && tile_n == 0 && t == 0) put_range(range, tile_m, mn, mx);
  RangeView view(tiles_m);
  for (int polls = range.polls;; polls = 0) {
    if (t < kWave) {
      const int missing = tiles_m > 1 ? get_ranges(range, tiles_m, static_cast<int>(tile), polls, view, mn, mx) : -1;
      if (missing < 0) {
        double s;
        int32_t z;
        choose_qparams(mn, mx, 0, 255, reduce_range != 0, &s, &z);
        if (t == 0) {
          s_scale = static_cast<float>(s);
          s_inv = 1.0f / static_cast<float>(s);  // IEEE division, as the separate quantize kernels
          s_zp = static_cast<float>(z);
        }
      }
      if (t == 0) s_missing = missing;
    }
    __syncthreads();
    const int missing = s_missing;
    if (missing < 0) break;
    // Those rows' block has not run yet, or not for this long: their range, read here.
    mn = __builtin_inff();
    mx = -__builtin_inff();
    const int64_t first = static_cast<int64_t>(missing) * BM, last = a.M - 1;
#pragma unroll 1
    for (int k = 4 * lane; k < K; k += 4 * kWave) {
      v4f v[BM / WAVES];
#pragma unroll
      for (int j = 0; j < BM / WAVES; ++j) {  // (rows past M: the last one again)
        const int64_t row = first + wave_u + j * WAVES;
        v[j] = reinterpret_cast<const FourFloats*>(x + (row < last ? row : last) * ldx + (k + 4 <= K ? k : K - 4))->v;
      }
#pragma unroll
      for (int j = 0; j < BM / WAVES; ++j) take_four(v[j], mn, mx);
    }
    block_range<WAVES>(mn, mx, s_range, t);
    if (t == 0) put_range(range, missing, mn, mx);
    if (t < kWave) view.add(missing, mn, mx);
    __syncthreads();                         // (s_missing is written again)
  }

  // ---- codes into the wave's LDS, without the sign of unsigned bytes; zeros behind K
  const float inv = s_inv, zp_f = s_zp;
  const XQuant xq{s_scale, 128 - static_cast<int>(zp_f)};
  const auto swizzle = [](int row) { return (row / (16 / kSlots)) & (kSlots - 1); };
  uint8_t* const mine = &sX[wave_u][0];
  {
    const int past = c + 4 - K;              // values of the group that are the row's own last ones
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = i * kRows + lane / kLanes, at = lane % kLanes;
      uint32_t q = fused_codes(held[i], inv, zp_f);
      if (past > 0) q >>= 8 * (past & 3);
      q = past >= 4 ? 0u : q ^ 0x80808080u;
      *reinterpret_cast<uint32_t*>(mine + r * S + (((at >> 2) ^ swizzle(r)) << 4) + 4 * (at & 3)) = q;
    }
  }
  wave_sync_lds();
  v16i acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[ct][r] = 0;
#pragma unroll
  for (int j = 0; j < kSteps; ++j) {
    const v4i xv = ld16(mine + li * S + (((2 * j + half) ^ swizzle(li)) << 4));
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[ct][j], xv, acc[ct], 0, 0, 0);
  }
  wave_sync_lds();
  if (t < BN) {
    s_raw[0][t] = colsum;
    s_raw[1][t] = scale;
    s_raw[2][t] = bias;
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const v4i part = {acc[ct][4 * g], acc[ct][4 * g + 1], acc[ct][4 * g + 2], acc[ct][4 * g + 3]};
      *reinterpret_cast<v4i*>(mine + li * kRedPitch + (32 * ct + 8 * g + 4 * half) * 4) = part;
    }
  __syncthreads();
#pragma unroll
  for (int idx = t; idx < BM * BN / 4; idx += WAVES * kWave)
    ksplit_finish_four<kOutF32, BN, WAVES>(a, &sX[0][0], kWaveLds, s_raw, xq, m0, n0, idx);
}

}  // namespace tmq
