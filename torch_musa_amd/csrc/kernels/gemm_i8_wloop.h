// int8 MFMA GEMM for grids smaller than the chip and K beyond what fits LDS at once (gfx950): tiles of 32 rows x 32 or 64
// channels whose eight waves split K, each walking its share in pieces through registers, with no barrier before the partial
// tiles meet.
//
// What bounds these products is what a CU pulls from the L2s, 100 to 110 bytes a nanosecond here where few tiles share them
// (a loop of copies alone reaches 120 to 150 where an XCD's CUs read the same lines), and before that how
// much of it is on its way: the pipelined tiles of gemm_i8_core.h request a 64-byte stage at a time for all waves
// behind one barrier (M = 174, N = 1088, K = 4544 on 51 tiles of 64 x 64 with two wave groups: 0.14 us a stage).
// Here a wave holds two pieces of both operands: 256 bytes of K by 32 rows and 32 channels, or 128 bytes by 32 and 64: 16
// (12) requests of 1 KB each, 256 (192) KB a CU in flight.  A piece's activations go to the wave's own LDS (whole
// lines of a row per request, the MFMA layout back out), its weights stay in registers in the packed layout, and as soon
// as it has been multiplied the piece after the next is requested into the same registers.
// The sign flip of unsigned activations and the zeros behind K are applied on the way into LDS.
// A wave's pieces are every eighth one and not a run of its own, and nothing is requested that is not multiplied: with runs,
// and the pieces past a wave's last fetched again so that every turn of the loop was alike, 482 x 5232 -> 768 took 12.6 us for
// 10.1 now, 1437 x 5184 -> 256 12.6 | 10.3, 76 x 5824 -> 128 8.9 | 7.2, 196 x 2304 -> 256 7.0 | 4.6 (of 266 x 6592 -> 1600's 13.4 ->
// 10.7 us the order alone is 1.0: rows off the 128-byte grid share a line between neighbouring pieces).
//
// Measured (us, weights from memory, the best other kernel | this one): M = 56, N = 1920, K = 4752 12.8 | 8.4; M = 63, N = 107,
// K = 5376 11.5 | 7.4; M = 407, N = 154, K = 6080 10.9 (its former self) | 8.2; M = 364, N = 320, K = 11968 24.7 | 14.8 before.
// RAGGED: rows of any K >= 16, pitch and address are read where they lie, by requests of any alignment; a row's last chunk as its
// last 16 bytes, shifted to their place.  On a round of tiles that beats staging them for 64 x 64 tiles, whose chain of stages is
// as long as K, and the copy onto the grid with its launch (us, those | these: 39 x 1098 -> 64 6.1 | 4.3, 137 x 1246 -> 203 6.9 | 4.7,
// 244 x 2680 -> 266 9.5 | 5.0, 1523 x 2982 -> 72 10.7 | 6.2, 542 x 745 -> 945 6.0 | 4.7, 50 x 270 -> 88 4.0 | 3.5, 71 x 7470 -> 512
// 11.1 | 10.6, 1073 x 5823 -> 320 18.2 | 13.1).  Beyond one round the larger tiles are ahead: 517 x 2051 -> 1000 8.9 | 10.5.
// XConvTable: a convolution's windows.  One thread a row works out where its window lies and which taps are inside the image, two
// divisions a piece give a lane its chunk's tap, and the zero point goes in for what is outside on the way into LDS: no table of
// the k order, no barrier but the one behind the windows.  Pieces of 128 bytes here also for 32 channels a tile (with 256 the row
// offsets and masks left 11 registers in memory).  conv_waves_tile (conv2d.hip) has what it is worth.
//
// Tried: 64 x 64 tiles the same way (256 registers; 273 x 5760 -> 2432 14.0 against 13.9 for lone 64 x 64 tiles in a ring of six
// stages, 482 x 5232 -> 768 14.4); K split over two to sixteen blocks as well, the last to arrive adding the others' partial sums
// (51 x 8384 -> 256 8.5 -> 7.9 with three, otherwise level or behind: the sums' way through memory costs 2.5 us); off the
// grid 517 x 1000 -> 2051 11.0 against 7.8); tiles of four waves, two blocks a CU, where there are more than 256 (1445 x 1472 -> 288 6.9
// against 5.9 for 32 x 64 tiles of eight).
#pragma once

#include "gemm_i8_onepass.h"

namespace tmq {

constexpr int kWloopWaves = 8;

// What the epilogue reads of the kernel's arguments, into scalar registers: called with a wave's requests on their way, so that
// the argument buffer's latency passes under theirs and not behind the last barrier.
__device__ __forceinline__ GemmArgs epilogue_args(const GemmArgs& a) {
  GemmArgs e = a;
  asm volatile("" : "+s"(e.M), "+s"(e.N), "+s"(e.bias), "+s"(e.w_scale_stride), "+s"(e.out_scale), "+s"(e.zp_f), "+s"(e.lo_f),
                    "+s"(e.hi_f), "+s"(e.y), "+s"(e.ldy), "+s"(e.n_off), "+s"(e.f_kind));
  return e;
}

// Tiles of 32 rows x 32 CT channels, PB bytes of K a piece.
template <int MODE, int CT, class XSRC = XLinear>
__global__ __launch_bounds__(kWloopWaves* kWave, 2) void gemm_i8_wloop_kernel(GemmArgs a, XSRC xs) {
  constexpr bool kConv = std::is_same<XSRC, XConvTable>::value, RAGGED = std::is_same<XSRC, XLinearRagged>::value;
  constexpr int BM = 32, BN = 32 * CT, PB = kConv ? 128 : 256 / CT, WAVES = kWloopWaves;
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
  // this wave's pieces: every eighth, so that neighbouring ones, which share the lines that rows off the 128-byte grid
  // have at a piece's ends, are asked for together
  int p = wave_u, left = wave_u < pieces ? (pieces - wave_u + WAVES - 1) / WAVES : 0;

  const uint8_t* xtile;
  const int slot = lane % kLPR;
  uint32_t xrow[kNX];
  uint64_t inside[kNX];                      // (convolutions) XLoader<XConvTable>
  if constexpr (kConv) {
    // the windows of the tile's rows, one thread each: offset of the corner from the tile's first image, taps inside the image
    struct Window {
      uint32_t off, unused;
      uint64_t inside;
    };
    __shared__ Window s_window[BM];
    const uint32_t image = static_cast<uint32_t>(m0) / static_cast<uint32_t>(xs.OH * xs.OW);
    xtile = xs.x + static_cast<int64_t>(image) * xs.H * xs.W * xs.IC + xs.ic_off;
    if (t < BM) {
      XLoader<XConvTable> row;
      row.init(xs, m0 + t, a.M);
      s_window[t] = Window{static_cast<uint32_t>(row.img - xtile) + static_cast<uint32_t>(row.off0), 0, row.inside};
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kNX; ++i) {
      xrow[i] = s_window[i * kRPL + lane / kLPR].off;
      inside[i] = s_window[i * kRPL + lane / kLPR].inside;
    }
  } else {
    xtile = xs.x + m0 * xs.ldx;
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
    uint32_t outside;                        // (convolutions) bit i: x[i] lies outside the image
  };
  // (chunks past K: bytes of the row, zeroed below)
  const auto request = [&](int p, Piece& pc) {
    __builtin_amdgcn_sched_barrier(0);
    const int c = p * kLPR + slot;
    if constexpr (kConv) {
      // (chunks past K: no tap)
      const uint32_t tap = c < KC ? static_cast<uint32_t>(c) / static_cast<uint32_t>(xs.icb) : kConvMaxTaps;
      const int kh = static_cast<int>(tap / static_cast<uint32_t>(xs.KW));
      const uint32_t off = static_cast<uint32_t>(
          (kh * xs.dil_h * xs.W + (static_cast<int>(tap) - kh * xs.KW) * xs.dil_w) * xs.IC + (c - static_cast<int>(tap) * xs.icb) * 16);
      pc.outside = 0;
#pragma unroll
      for (int i = 0; i < kNX; ++i) {
        const uint32_t in = static_cast<uint32_t>(inside[i] >> tap) & 1u;
        pc.outside |= (in ^ 1u) << i;
        pc.x[i] = ld16(xtile + ((xrow[i] + off) & (0u - in)));
      }
    } else if constexpr (RAGGED) {
      const uint32_t off = static_cast<uint32_t>(16 * c + 16 <= K ? 16 * c : K - 16);
#pragma unroll
      for (int i = 0; i < kNX; ++i) pc.x[i] = ld16_any(xtile + (xrow[i] + off));
    } else {
      const uint32_t off = static_cast<uint32_t>(c < KC ? c : KC - 1) * 16u;
#pragma unroll
      for (int i = 0; i < kNX; ++i) pc.x[i] = ld16(xtile + (xrow[i] + off));
    }
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int kc = p * kLPR + 2 * j + half;
      const int64_t woff = static_cast<int64_t>(kc < kc_last ? kc : kc_last) * 256;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) pc.w[ct][j] = ld16(wlane[ct] + woff);
    }
    __builtin_amdgcn_sched_barrier(0);
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
    const int keep = (RAGGED ? 16 * c < K : c < KC) ? -1 : 0;
    if (RAGGED && p == pieces - 1) {         // (a row's last chunk was read where its last 16 bytes are)
      const int past = 16 * c - (K - 16);
#pragma unroll
      for (int i = 0; i < kNX; ++i) pc.x[i] = shift_down_bytes(pc.x[i], past > 0 && past < 16 ? past : 0);
    }
#pragma unroll
    for (int i = 0; i < kNX; ++i) {
      const int r = i * kRPL + lane / kLPR;
      v4i v = pc.x[i];
      if constexpr (kConv) {
        const int pad = static_cast<int>(xs.pad_word);
        if ((pc.outside >> i) & 1u) v = v4i{pad, pad, pad, pad};
      }
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
  // Straight code for the pieces that are left, so that nothing is fetched that is not multiplied and the compiler knows
  // how many requests are behind the one it waits for.
  constexpr int kNext = WAVES;
  XQuant xq;
  GemmArgs e;
  const auto arguments = [&] {
    xq = x_quant(a);
    e = epilogue_args(a);
  };
  if (left >= 2) {
    request(p, pc[0]);
    request(p + kNext, pc[1]);
    arguments();
    for (; left >= 4; left -= 2, p += 2 * kNext) {
      multiply(p, pc[0]);
      request(p + 2 * kNext, pc[0]);
      multiply(p + kNext, pc[1]);
      request(p + 3 * kNext, pc[1]);
    }
    multiply(p, pc[0]);
    if (left == 3) {
      request(p + 2 * kNext, pc[0]);
      multiply(p + kNext, pc[1]);
      multiply(p + 2 * kNext, pc[0]);
    } else {
      multiply(p + kNext, pc[1]);
    }
  } else {
    if (left == 1) request(p, pc[0]);
    arguments();
    if (left == 1) multiply(p, pc[0]);
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
    ksplit_finish_four<MODE, BN, WAVES, kConv>(e, &sX[0][0], kWaveLds, s_raw, xq, m0, n0, idx);
}

}  // namespace tmq
