// quantized::conv2d over images of three channels (gfx950): the first layer of an image network
// (3 -> 64 channels, 7 x 7, stride 2), one group, no dilation.
//
// The scheme of conv_runs.h -- k ordered (kernel row, run of the row's taps), weights of 64 (32)
// output channels in registers for the whole launch, a lane ends up with 4 NT consecutive channels
// of one pixel -- with one change: in LDS a pixel is four bytes, the fourth meeting zero weights.
// A run is then KW * 4 bytes, padded to RP = a multiple of 16, and an operand always starts on a
// dword (with an even stride on two), so it is one or two LDS instructions at an address of one
// addition; packed as three bytes it starts anywhere and is five dwords put together by four
// v_alignbyte at an address of six operations.  The fourth byte costs nothing: rows are padded to
// 16 bytes anyway (7 taps: 21 or 28 bytes, both 32).  The copy into LDS moves groups of four pixels,
// twelve bytes of the image at any alignment, whose pixels outside the image are the zero point, so
// padding needs no pass of its own; the next tile's groups are on their way while a tile is multiplied.
// The requantisation multipliers and bias terms of the lane's channels stay in registers like the weights.
//
// What bounds it is the length of one block's chain.  [32, 3, 224, 224] -> 64 channels, 7 x 7 stride 2 (30.5 MB, 4.7 us at
// the rate of a copy) takes 17.0 us, 20.5 us with the byte runs of conv_runs.h.  Its 736 tiles of five rows are one per
// block, and the chip holds all blocks at once: no second tile runs under the waits of the first, so set-up, first loads,
// LDS, products and stores follow one another.  Counters: the waves wait in 39 % of their cycles (for an issue slot in
// another 26 %) and issue vector instructions in 22 %, at three waves a SIMD.  Of those 4.0 M instructions 1.6 M requantise
// (four a value), 0.4 M are products, 0.4 M are addresses and operands of the pieces, and 1.6 M are the waves' set-up,
// 550 each: positions and edge tests of the first groups, weights, constants.
#pragma once

#include "conv_runs.h"

namespace tmq {

constexpr int kCiUnits = 4;  // groups of four pixels a thread holds for the next tile

// One 16-byte slot of the weight layout: conv_runs_slot for runs of four-byte pixels.
__device__ __forceinline__ v4i conv_image_slot(const int8_t* __restrict__ w, int64_t slot, int OC, int KH, int KW,
                                               int RP, int KS) {
  const int NT = conv_runs_tiles(OC);
  const int lane = static_cast<int>(slot & 63);
  const int64_t op = slot >> 6;
  const int ks = static_cast<int>(op % KS), nt = static_cast<int>((op / KS) % NT);
  const int64_t cb = op / (NT * KS);
  const int i = lane & 15;
  const int64_t n = cb * 16 * NT + 4 * NT * (i >> 2) + 4 * nt + (i & 3);
  const int k = 64 * ks + 16 * (lane >> 4);
  const int kh = k / RP, ro = k - kh * RP;
  uint32_t words[4] = {0, 0, 0, 0};
  if (n < OC && kh < KH)
    for (int p = 0; p < 4; ++p)
      if (ro / 4 + p < KW)
        for (int c = 0; c < 3; ++c)
          words[p] |= static_cast<uint32_t>(static_cast<uint8_t>(w[((n * KH + kh) * KW + ro / 4 + p) * 3 + c])) << (8 * c);
  return v4i{static_cast<int>(words[0]), static_cast<int>(words[1]), static_cast<int>(words[2]),
             static_cast<int>(words[3])};
}

// EVEN: the horizontal stride is even (operands on 8 bytes).  a.pitch: LDS bytes per staged row, 16 per group.
// KSN: k-steps of the loop, at least KS (the weights of the others are zero).
template <int MODE, int POST, int NT, int KSN, bool EVEN, bool PLAIN = false>
__global__ __launch_bounds__(kCrThreads, 3) void conv_image_kernel(ConvRunArgs a) {
  constexpr int kCrBN = 16 * NT;   // output channels per block (grid y)
  constexpr int kLaneCh = 4 * NT;  // consecutive channels of one pixel in a lane
  extern __shared__ __attribute__((aligned(16))) uint8_t sX[];  // staged image rows
  __shared__ __attribute__((aligned(16))) int s_acc0[kCrBN];
  __shared__ __attribute__((aligned(16))) float s_mult[kCrBN];
  __shared__ __attribute__((aligned(16))) float s_bdiv[kCrBN];
  const int t = threadIdx.x, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int pj = lane & 15, pq = lane >> 4;
  const int n0 = static_cast<int>(blockIdx.y) * kCrBN;
  const int KS = a.KS;

  // ---- the copy: unit u of a tile = group u % G of staged row u / G
  const int G = a.pitch >> 4, units = a.rows_in * G;
  const int64_t x_bytes = static_cast<int64_t>(a.B) * a.H * a.W * 3;
  struct __attribute__((packed, aligned(1))) Twelve {
    uint32_t d[3];
  };
  int ur[kCiUnits], uc[kCiUnits];  // this thread's units: staged row and first pixel in it (the same in every tile)
#pragma unroll
  for (int i = 0; i < kCiUnits; ++i) {
    const int u = t + i * kCrThreads;
    ur[i] = u < units ? u / G : -1;
    uc[i] = (u - (u / G) * G) * 4;
  }
  Twelve pre[kCiUnits];
  struct TilePos {
    int b, oh0, ow0;
  };
  const auto tile_pos = [&](uint32_t tile) {
    TilePos tp;
    const uint32_t trb = tile / static_cast<uint32_t>(a.tiles_w);
    tp.ow0 = static_cast<int>(tile - trb * static_cast<uint32_t>(a.tiles_w)) * a.TW;
    tp.b = static_cast<int>(trb / static_cast<uint32_t>(a.tiles_h));
    tp.oh0 = (static_cast<int>(trb) - tp.b * a.tiles_h) * a.TR;
    return tp;
  };
  const auto request = [&](const TilePos& tp) {
#pragma unroll
    for (int i = 0; i < kCiUnits; ++i) {
      const int ih = tp.oh0 * a.sh - a.ph + ur[i], iw = tp.ow0 * a.sw - a.pw + uc[i];
      if (ur[i] < 0 || static_cast<unsigned>(ih) >= static_cast<unsigned>(a.H) || iw + 4 <= 0 || iw >= a.W) continue;
      const int64_t o = ((static_cast<int64_t>(tp.b) * a.H + ih) * a.W + iw) * 3;
      const int64_t at = o < 0 ? 0 : o + 12 > x_bytes ? x_bytes - 12 : o;  // (the host: at least twelve bytes)
      pre[i] = *reinterpret_cast<const Twelve*>(a.x + at);
      if (at != o) {  // over the tensor's first or last byte
        const v4i v = {static_cast<int>(pre[i].d[0]), static_cast<int>(pre[i].d[1]), static_cast<int>(pre[i].d[2]), 0};
        const v4i m = at > o ? shift_up_bytes(v, static_cast<int>(at - o)) : shift_down_bytes(v, static_cast<int>(o - at));
        pre[i] = Twelve{{static_cast<uint32_t>(m.x), static_cast<uint32_t>(m.y), static_cast<uint32_t>(m.z)}};
      }
    }
  };
  const auto store_tile = [&](const TilePos& tp) {
    const uint32_t flip = a.x_xor, pad = a.pad_word ^ a.x_xor;
#pragma unroll
    for (int i = 0; i < kCiUnits; ++i) {
      if (ur[i] < 0) continue;
      const int ih = tp.oh0 * a.sh - a.ph + ur[i], iw = tp.ow0 * a.sw - a.pw + uc[i];
      const bool row_in = static_cast<unsigned>(ih) < static_cast<unsigned>(a.H);
      const uint32_t d0 = pre[i].d[0] ^ flip, d1 = pre[i].d[1] ^ flip, d2 = pre[i].d[2] ^ flip;
      // three-byte pixels to dwords; the fourth byte is whatever follows
      uint32_t p[4] = {d0, __builtin_amdgcn_alignbyte(d1, d0, 3), __builtin_amdgcn_alignbyte(d2, d1, 2), d2 >> 8};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        p[j] = row_in && static_cast<unsigned>(iw + j) < static_cast<unsigned>(a.W) ? p[j] : pad;
      *reinterpret_cast<v4i*>(sX + ur[i] * a.pitch + uc[i] * 4) =
          v4i{static_cast<int>(p[0]), static_cast<int>(p[1]), static_cast<int>(p[2]), static_cast<int>(p[3])};
    }
  };
  TilePos cur{};
  if (static_cast<int>(blockIdx.x) < a.tiles) {
    cur = tile_pos(blockIdx.x);
    request(cur);
  }
  // ---- weights and constants
  v4i wreg[NT][KSN];
  {
    const uint8_t* const wsrc = a.w_runs + (static_cast<int64_t>(blockIdx.y) * NT * KS * kWave + lane) * 16;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int ks = 0; ks < KSN; ++ks)
        wreg[nt][ks] = ks < KS ? ld16(wsrc + (nt * KS + ks) * (kWave * 16)) : v4i{0, 0, 0, 0};
  }
  if (t < kCrBN) {
    const int n = n0 + t;
    int acc0 = 0;
    float mult = 0.f, bdiv = 0.f;
    if (n < a.OC) {
      acc0 = a.acc_coef * a.colsum[n];
      if constexpr (MODE != kOutAcc32) {
        const float atw = a.x_scale * a.w_scales[n * a.w_scale_stride];
        mult = atw / a.out_scale;
        bdiv = a.bias != nullptr ? bias_term(a.w_scale_stride == 0, a.bias[n], atw) : 0.f;
      }
    }
    s_acc0[t] = acc0;
    s_mult[t] = mult;
    s_bdiv[t] = bdiv;
  }
  float bmul = 1.0f;
  if constexpr (MODE != kOutAcc32) bmul = bias_mul(a.w_scale_stride == 0, a.x_scale * a.w_scales[0]);
  // this lane's piece of every k-step: kernel row and byte inside the run
  int lk[KSN];
#pragma unroll
  for (int ks = 0; ks < KSN; ++ks) {
    const int koff = ks * 64 + pq * 16;
    int kh = koff / a.RP, ro = koff - kh * a.RP;
    if (kh >= a.KH) {  // past the last kernel row: zero weights, any staged bytes
      kh = a.KH - 1;
      ro = 0;
    }
    lk[ks] = kh * a.pitch + ro;
  }
  __syncthreads();
  float mult[kLaneCh], bdiv[kLaneCh];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int at = kLaneCh * pq + 4 * nt;
    const v4f m = *reinterpret_cast<const v4f*>(&s_mult[at]), b = *reinterpret_cast<const v4f*>(&s_bdiv[at]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mult[4 * nt + r] = m[r];
      bdiv[4 * nt + r] = b[r];
    }
  }
  const int cb = n0 + kLaneCh * pq;
  const bool residual = POST == 1 || (POST == 2 && a.post.accum != nullptr);

  const int tile_mt = a.TR * a.mtw;
  for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    const TilePos here = cur;
    store_tile(here);
    __syncthreads();
    if (tile + static_cast<int>(gridDim.x) < a.tiles) {
      cur = tile_pos(static_cast<uint32_t>(tile) + gridDim.x);
      request(cur);
    }
    // ---- multiply: 16 pixels of one output row per wave and turn
    const int tw_valid = a.OW - here.ow0 < a.TW ? a.OW - here.ow0 : a.TW;
    const int th_valid = a.OH - here.oh0 < a.TR ? a.OH - here.oh0 : a.TR;
    const int64_t opix0 = (static_cast<int64_t>(here.b) * a.OH + here.oh0) * a.OW + here.ow0;
    int orow = 0, mcol = wave;  // this wave's piece: row of the tile, 16-pixel piece of the row
    for (int mt = wave; mt < tile_mt; mt += kCrWaves, mcol += kCrWaves) {
      while (mcol >= a.mtw) {
        mcol -= a.mtw;
        ++orow;
      }
      if (orow >= th_valid || mcol * 16 >= tw_valid) continue;  // (the same for the whole wave)
      const int pcol = mcol * 16 + pj;
      const int pc = pcol < tw_valid ? pcol : tw_valid - 1;
      const int64_t off = (opix0 + static_cast<int64_t>(orow) * a.OW + pcol) * a.OC + cb;
      const bool live = pcol < tw_valid && cb < a.OC;
      RunsResidual<NT> accw{};
      if (residual && live) accw = runs_residual<NT>(a, off, cb);
      const uint8_t* const src = sX + orow * a.sh * a.pitch + pc * a.sw * 4;
      v4i acc[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = *reinterpret_cast<const v4i*>(&s_acc0[kLaneCh * pq + 4 * nt]);
#pragma unroll
      for (int ks = 0; ks < KSN; ++ks) {
        {
          v4i xv;
          if constexpr (EVEN) {
            const v2i* const p = reinterpret_cast<const v2i*>(src + lk[ks]);
            const v2i lo = p[0], hi = p[1];
            xv = v4i{lo.x, lo.y, hi.x, hi.y};
          } else {
            const int* const p = reinterpret_cast<const int*>(src + lk[ks]);
            xv = v4i{p[0], p[1], p[2], p[3]};
          }
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[nt][ks], xv, acc[nt], 0, 0, 0);
        }
      }
      if (live) runs_requant_store<MODE, POST, NT, PLAIN>(a, acc, off, cb, mult, bdiv, bmul, accw, a.through != 0);
    }
    __syncthreads();  // the staged rows are overwritten by the next tile
  }
}

}  // namespace tmq
