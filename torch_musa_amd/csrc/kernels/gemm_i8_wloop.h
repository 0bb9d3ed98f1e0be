// int8 MFMA GEMM for grids smaller than the chip against a long K (gfx950): tiles of 32 rows x 32 or 64 channels whose
// eight waves split K, each walking its share in pieces through registers, with no barrier before the partial tiles meet.
//
// What bounds these products is what a CU pulls from the L2s and memory, about 60 bytes a nanosecond, and before that how
// much of it is on its way: the pipelined tiles of gemm_i8_core.h request a 64-byte stage at a time for all waves
// behind one barrier (M = 174, N = 1088, K = 4544 on 51 tiles of 64 x 64 with two wave groups: 0.14 us a stage), and the kernels that
// have all of a wave's share in registers and LDS at once (gemm_i8_wstream_kernel, gemm_i8_wring_kernel) end at K = 4096.
// Here a wave holds two pieces of both operands: 256 bytes of K by 32 rows and 32 channels, or 128 bytes by 32 and 64: 16
// (12) requests of 1 KB each, 256 (192) KB a CU in flight.  A piece's activations go to the wave's own LDS (whole
// lines of a row per request, the MFMA layout back out), its weights stay in registers in the packed layout, and as soon
// as it has been multiplied the piece after the next is requested into the same registers.
// The sign flip of unsigned activations and the zeros behind K are applied on the way into LDS.
//
// Measured (us, weights from memory, the best other kernel | this one): M = 174, N = 1088, K = 4544 12.5 | 8.6;
// M = 102, N = 1280, K = 6784 16.2 | 10.1; M = 267, N = 256, K = 8704 19.6 | 10.3; M = 364, N = 320, K = 11968 24.7 | 14.8.
// At those a block pulls 64 K bytes at 48 ... 60 bytes a nanosecond behind 2 us of launch and first bytes.  Tried: 64 x 64
// tiles the same way (never the best: M = 561, N = 1920, K = 6528 33 against 27); rows off the 16-byte grid read where
// they lie (M = 1633, N = 163, K = 5834 20.9 against 17.2 for the tiles that stage them), which are copied onto the grid
// instead; 32 x 32 tiles of four waves, two blocks a CU, where there are more than 256 (M = 2129, N = 192, K = 7104 21.9
// against 15.6 for 32 x 64 tiles of eight).
#pragma once

#include "gemm_i8_onepass.h"

namespace tmq {

constexpr int kWloopWaves = 8;

// Tiles of 32 rows x 32 CT channels, PB bytes of K a piece.
template <int MODE, int CT>
__global__ __launch_bounds__(kWloopWaves* kWave, 2) void gemm_i8_wloop_kernel(GemmArgs a, XLinear xs) {
  constexpr int BM = 32, BN = 32 * CT, PB = 256 / CT, WAVES = kWloopWaves;
  constexpr int kLPR = PB / 16;              // 16-byte chunks (lanes) of a row in a piece
  constexpr int kRPL = kWave / kLPR;         // rows per request
  constexpr int kNX = BM / kRPL;             // activation requests of a piece
  constexpr int kSteps = PB / 32;            // k-steps of a piece
  constexpr int kRedPitch = BN * 4 + 16;
  constexpr int kWaveLds = BM * PB > BM * kRedPitch ? BM * PB : BM * kRedPitch;  // a piece's activations, then the partial tile
  __shared__ __attribute__((aligned(16))) uint8_t sX[WAVES][kWaveLds];
  __shared__ __attribute__((aligned(16))) int s_raw[3][kWave];  // colsum, weight scale, bias as fetched

  const int t = threadIdx.x, lane = t % kWave;
  const int wave_u = __builtin_amdgcn_readfirstlane(t / kWave);
  const int li = lane & 31, half = lane >> 5;
  const TileAt at = tile_of_block<BM, BN, true>(a);
  const int64_t m0 = at.m0, n0 = at.n0;
  const int K = static_cast<int>(a.K);
  const int KC = K >> 4;                     // 16-byte chunks of a row (K is a multiple of 16)
  const int pieces = (K + PB - 1) / PB;
  // this wave's pieces: an equal run of them
  const int each = pieces / WAVES, more = pieces - each * WAVES;
  const int first = wave_u * each + (wave_u < more ? wave_u : more);
  const int last = first + each + (wave_u < more ? 1 : 0);

  const uint8_t* const xtile = xs.x + m0 * xs.ldx;
  const int slot = lane % kLPR;
  uint32_t xrow[kNX];
  {
    const int64_t m_last = a.M - 1 - m0;     // rows past M: clamped, never stored
#pragma unroll
    for (int i = 0; i < kNX; ++i) {
      const int r = i * kRPL + lane / kLPR;
      xrow[i] = static_cast<uint32_t>((r < m_last ? r : m_last) * xs.ldx);
    }
  }
  const int kc_last = static_cast<int>(a.w_kchunks) - 1;
  const uint8_t* wlane[CT];
  {
    const int64_t nb_last = ceil_div(a.N, 16) - 1 - n0 / 16;  // 16-row blocks past N: clamped, never stored
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int64_t rb0 = 2 * ct + ((lane >> 4) & 1);
      wlane[ct] = a.w_packed + (n0 / 16 + (rb0 < nb_last ? rb0 : nb_last)) * a.w_kchunks * 256 + (lane & 15) * 16;
    }
  }
  struct Piece {
    v4i x[kNX], w[CT][kSteps];
  };
  // (pieces past this wave's last fetch that one again and are not multiplied; chunks past K: bytes of the row, zeroed below)
  const auto request = [&](int p, Piece& pc) {
    const int pp = p < last ? p : last > 0 ? last - 1 : 0;
    const int c = pp * kLPR + slot;
    const uint32_t off = static_cast<uint32_t>(c < KC ? c : KC - 1) * 16u;
#pragma unroll
    for (int i = 0; i < kNX; ++i) pc.x[i] = ld16(xtile + (xrow[i] + off));
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int kc = pp * kLPR + 2 * j + half;
      const int64_t woff = static_cast<int64_t>(kc < kc_last ? kc : kc_last) * 256;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) pc.w[ct][j] = ld16(wlane[ct] + woff);
    }
  };
  // (the tile's constants first: nothing behind them is waited for when they are put down at the end)
  const int64_t n_raw = (n0 + t % BN < a.N ? n0 + t % BN : a.N - 1) + a.n_off;
  const int colsum = a.colsum[n_raw];
  int scale = 0, bias = 0;
  if constexpr (MODE != kOutAcc32) {  // (raw accumulators: the caller passes no scales)
    scale = __float_as_int(a.w_scales[n_raw * a.w_scale_stride]);
    bias = __float_as_int((a.bias != nullptr ? a.bias : a.w_scales)[a.bias != nullptr ? n_raw : 0]);
  }
  Piece pc[2];
  __builtin_amdgcn_sched_barrier(0);
  request(first, pc[0]);
  __builtin_amdgcn_sched_barrier(0);
  request(first + 1, pc[1]);
  __builtin_amdgcn_sched_barrier(0);
  v16i acc[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[ct][r] = 0;

  // slots of a row in LDS, so that the lanes of a read (32 rows, one chunk) lie in different banks
  const auto swizzle = [](int row) { return kLPR == 16 ? row & 15 : (row >> 1) & 7; };
  uint8_t* const mine = &sX[wave_u][0];
  const int flip = static_cast<int>(a.x_xor);
  const auto multiply = [&](int p, Piece& pc) {
    const int c = p * kLPR + slot;
#pragma unroll
    for (int i = 0; i < kNX; ++i) {
      const int r = i * kRPL + lane / kLPR;
      v4i v = pc.x[i];
      const int keep = c < KC && p < last ? -1 : 0;
      v = (v ^ v4i{flip, flip, flip, flip}) & v4i{keep, keep, keep, keep};
      *reinterpret_cast<v4i*>(mine + r * PB + ((slot ^ swizzle(r)) << 4)) = v;
    }
    wave_sync_lds();
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const v4i xv = ld16(mine + li * PB + (((2 * j + half) ^ swizzle(li)) << 4));
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[ct] = __builtin_amdgcn_mfma_i32_32x32x32_i8(pc.w[ct][j], xv, acc[ct], 0, 0, 0);
    }
    wave_sync_lds();                         // (the next piece is written over this one)
  };
  // (both pieces in every turn, an odd last one with zeros: the counts of outstanding requests stay exact)
  for (int p = first; p < last; p += 2) {
    multiply(p, pc[0]);
    __builtin_amdgcn_sched_barrier(0);
    request(p + 2, pc[0]);
    __builtin_amdgcn_sched_barrier(0);
    multiply(p + 1, pc[1]);
    __builtin_amdgcn_sched_barrier(0);
    request(p + 3, pc[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (t < BN) {
    s_raw[0][t] = colsum;
    s_raw[1][t] = scale;
    s_raw[2][t] = bias;
  }
  // ---- the partial tile of this wave, over its own activations: a lane holds channels 32 ct + 8 g + 4 half + j
  // (g, j < 4) of row li
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
    ksplit_finish_four<MODE, BN, WAVES>(a, &sX[0][0], kWaveLds, s_raw, m0, n0, idx);
}

}  // namespace tmq
