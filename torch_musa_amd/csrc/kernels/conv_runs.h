// quantized::conv2d for a few input channels (gfx950): the first layer of an image
// network (3 -> 64 channels, 7 x 7, stride 2), pointwise layers whose channel count is
// no multiple of 16, one group, no dilation.
//
// With so few channels a 16-byte k-chunk of the MFMA cannot be "16 channels of one
// pixel".  In NHWC the KW taps of one kernel row are KW * IC *contiguous* bytes of an
// image row, so k is ordered (kh, run) with run = the RL = KW * IC bytes of a kernel
// row, padded to RP = a multiple of 16 with zero weights: the bytes an operand picks
// up past the run's end are multiplied by zero.  K = KH * RP is at most 256 here, the
// weights of 64 (32) output channels stay in registers (16 operands of
// v_mfma_i32_16x16x64_i8) for the whole launch; prepack lays them out per lane
// (conv_runs_slot) behind the packed weight of the other kernels.
//
// A block of four waves walks tiles of TR x TW output pixels of one image:
//   * it stages the (TR - 1) * stride + KH image rows the tile needs, as bytes, positions
//     outside the image as the activation zero point, sign flip of unsigned activations
//     applied.  The copy runs in aligned 16-byte loads whatever the address of an image
//     row: each staged row starts 0 ... 15 bytes before the tile's first byte of its row;
//   * a wave takes 16 output pixels of one output row at a time: the operand of pixel
//     p, kernel row kh, 16-byte piece c of the run is the 16 bytes at
//       row (orow * stride + kh), byte p * stride * IC + 16 c
//     of the staged rows -- any byte alignment, so it is put together from five aligned
//     words with v_alignbyte_b32;
//   * operand roles: weights are the rows (i), pixels the columns (j) of the MFMA,
//     D[i][j]: lane l, register r -> i = 4 (l / 16) + r, j = l % 16.  Row i of channel
//     tile nt (of NT = 4, or 2 for at most 32 output channels) is channel
//     4 NT (i / 4) + 4 nt + i % 4, so that a lane ends up with 4 NT consecutive channels of
//     one pixel: one 16-byte (8-byte) store.
// The x ^ 0x80 trick, the accumulator start value and the requantisation are those of
// gemm_i8_core.h.
#pragma once

#include "gemm_i8_core.h"
#include "tail_read.h"

namespace tmq {

constexpr int kCrThreads = 256;
constexpr int kCrWaves = kCrThreads / kWave;
constexpr int kCrMaxKS = 4;    // k-steps of 64 bytes
constexpr int kCrUnits = 4;    // 1 KB units of staged image rows per wave and tile: 16 KB per block

struct ConvRunArgs {
  const uint8_t* x;          // NHWC
  const uint8_t* w_runs;     // [channel block of 16 NT][channel tile nt][k-step][lane][16 B]: conv_runs_slot below
  const int32_t* colsum;
  const float* w_scales;
  const float* bias;
  void* y;
  int32_t tiles;             // B * tiles_h * tiles_w
  int B, H, W, IC, OH, OW, OC, KH, KW;
  int sh, sw, ph, pw;
  int RL, RP, KS;            // run bytes, padded run bytes, k-steps (KH * RP <= 64 KS)
  union {                    // (both sets side by side cost every pointwise layer 0.05 us more)
    struct {
      int TR, TW, mtw;       // output rows and columns per tile, 16-pixel pieces per tile row
      int rows_in, pitch;    // staged image rows, LDS bytes per staged row (multiple of 16)
      int tiles_h, tiles_w;
    };
    struct {                 // (pointwise) blockIdx -> XCD and place in it, blocks of an XCD's run (xcd_longer of the runs
                             // have one more), groups dealt to the XCDs
      uint32_t xcd_mask, xcd_shift, xcd_blocks, xcd_longer, deal_shift, deal_mask;
    };
  };
  union {
    int vec;                 // (int32 outputs) 16-byte stores per 4 channels are aligned
    int through;             // (bytes, conv_runs_kernel and conv_image_kernel) those of whole lanes: st16_through / st8_through
  };
  int whole;                 // (pointwise) pieces all of whose reads and stores lie inside the tensors
  int nblk, groups;          // (pointwise) channel blocks, and waves on each of them
  uint32_t nblk_magic;       // w / nblk = (w * nblk_magic) >> 32 for the waves w of the launch (nblk > 1)
  int32_t w_scale_stride;
  uint32_t x_xor, pad_word;  // pad_word: the activation zero point in 4 bytes, before the xor
  int32_t acc_coef;
  float x_scale, out_scale, zp_f, lo_f, hi_f;
  PostOps post;
};

// One 16-byte slot of the per-lane weight layout: slot index ->
// (channel block cb of 16 NT channels, channel tile nt, k-step ks, lane).  NT = 4 tiles per block,
// 2 for layers of at most 32 output channels.  The lane's row i = lane % 16 of tile nt is channel
// 16 NT cb + 4 NT (i / 4) + 4 nt + i % 4 (a lane of the kernel then holds 4 NT consecutive
// channels); its bytes are k = 64 ks + 16 (lane / 16) ... + 15 in (kh, run) order: kernel row
// kh = k / RP, byte k % RP of the run, which in OHWI weights is byte (kw, ic) = k % RP of the
// contiguous row w[n][kh][.][.]; zeros past the run's RL bytes, past the last kernel row and for
// channels that do not exist.
__host__ __device__ inline int conv_runs_tiles(int64_t OC) { return OC <= 32 ? 2 : 4; }
__device__ __forceinline__ v4i conv_runs_slot(const int8_t* __restrict__ w, int64_t slot, int OC, int KH, int RL,
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
  if (n < OC && kh < KH) {
    const int8_t* const src = w + (n * KH + kh) * RL;
    for (int b = 0; b < 16; ++b)
      if (ro + b < RL) words[b >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(src[ro + b])) << (8 * (b & 3));
  }
  return v4i{static_cast<int>(words[0]), static_cast<int>(words[1]), static_cast<int>(words[2]),
             static_cast<int>(words[3])};
}

struct __attribute__((packed, aligned(1))) U32AnyAlignment {
  uint32_t v;
};
// Requantise (or pass on) the 4 NT consecutive channels cb ... of one pixel that a lane holds after the
// MFMAs of its NT channel tiles, and store them at element offset `off` of the output: one store of 4 NT
// bytes where all the channels exist.  mult / bdiv: the constants of channel cb onwards.  PLAIN: the host found
// requant_plain_u8 to hold (zero point 0 for unsigned bytes, -128 for signed ones, no bounds inside the range).
// POST: 0 no post operations, 1 a residual and no SiLU, 2 SiLU (a residual if there is one); accw: the residual
// bytes of the lane's channels (runs_residual).
template <int NT>
struct RunsResidual {
  uint32_t w[NT];
};
template <int NT>
__device__ __forceinline__ RunsResidual<NT> runs_residual(const ConvRunArgs& a, int64_t off, int cb) {
  // one load of 4 NT bytes at any alignment where all the channels exist (a dword per four channels
  // took four requests, each waited for by itself)
  RunsResidual<NT> r;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) r.w[nt] = 0;
  const uint8_t* const src = a.post.accum + off;
  if (cb + 4 * NT <= a.OC) {
    if constexpr (NT == 4) {
      const v4i v = ld16_any(src);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) r.w[nt] = static_cast<uint32_t>(v[nt]);
    } else {
      const v2i v = reinterpret_cast<const V2iAnyAlignment*>(src)->v;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) r.w[nt] = static_cast<uint32_t>(v[nt]);
    }
  } else {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int left = a.OC - (cb + 4 * nt);
      if (left > 0) r.w[nt] = load_accum4(a.post, off + 4 * nt, left < 4 ? left : 4);
    }
  }
  return r;
}
template <int MODE, int POST, int NT, bool PLAIN>
__device__ __forceinline__ void runs_requant(const ConvRunArgs& a, const v4i (&acc)[NT], const float* mult_cb,
                                             const float* bdiv_cb, float bmul, const RunsResidual<NT>& accw,
                                             uint32_t (&packed)[NT]) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int raw[4] = {acc[nt][0], acc[nt][1], acc[nt][2], acc[nt][3]};
    const v4f mult = {mult_cb[4 * nt], mult_cb[4 * nt + 1], mult_cb[4 * nt + 2], mult_cb[4 * nt + 3]};
    const v4f bdiv = {bdiv_cb[4 * nt], bdiv_cb[4 * nt + 1], bdiv_cb[4 * nt + 2], bdiv_cb[4 * nt + 3]};
    if constexpr (POST != 0) {
      packed[nt] = requant4_post<MODE, POST, PLAIN>(raw, bdiv, bmul, mult, a.post, accw.w[nt], a.zp_f, a.lo_f, a.hi_f);
    } else {
      packed[nt] = requant4<MODE, true, PLAIN ? 1 : 0>(raw, bdiv, bmul, mult, a.zp_f, a.lo_f, a.hi_f);
    }
  }
}
// One store of a lane's 4 NT bytes, at any alignment (the same instruction as an aligned one); through: stores_through.h, dst
// on the grid of 4 NT bytes.
template <int NT>
__device__ __forceinline__ void runs_store(uint8_t* dst, const uint32_t (&packed)[NT], bool through) {
  if constexpr (NT == 4) {
    const v4i v = {static_cast<int>(packed[0]), static_cast<int>(packed[1]), static_cast<int>(packed[2]),
                   static_cast<int>(packed[3])};
    if (through) st16_through(dst, v);
    else st16_any(dst, v);
  } else {
    static_assert(NT == 2, "channel tiles per block: 2 or 4");
    if (through) st8_through(dst, (static_cast<uint64_t>(packed[1]) << 32) | packed[0]);
    else st8_any(dst, v2i{static_cast<int>(packed[0]), static_cast<int>(packed[1])});
  }
}
// A lane at the end of the channels, `left` of whose 4 NT exist: a word where four do, else bytes.
template <int NT>
__device__ __forceinline__ void runs_store_some(uint8_t* dst, const uint32_t (&packed)[NT], int left) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt, left -= 4) {
    if (left >= 4) {
      reinterpret_cast<U32AnyAlignment*>(dst + 4 * nt)->v = packed[nt];
    } else if (left > 0) {
      dst[4 * nt] = static_cast<uint8_t>(packed[nt]);
      if (left > 1) dst[4 * nt + 1] = static_cast<uint8_t>(packed[nt] >> 8);
      if (left > 2) dst[4 * nt + 2] = static_cast<uint8_t>(packed[nt] >> 16);
    }
  }
}
template <int MODE, int POST, int NT, bool PLAIN = false>
__device__ __forceinline__ void runs_requant_store(const ConvRunArgs& a, const v4i (&acc)[NT], int64_t off, int cb,
                                                   const float* mult_cb, const float* bdiv_cb, float bmul,
                                                   const RunsResidual<NT>& accw, bool through) {
  constexpr int kLaneCh = 4 * NT;
  if constexpr (MODE == kOutAcc32) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      int32_t* const dst = static_cast<int32_t*>(a.y) + off + 4 * nt;
      if (a.vec && cb + 4 * nt + 4 <= a.OC) {
        *reinterpret_cast<v4i*>(dst) = acc[nt];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (cb + 4 * nt + r < a.OC) dst[r] = acc[nt][r];
      }
    }
  } else {
    uint32_t packed[NT];
    runs_requant<MODE, POST, NT, PLAIN>(a, acc, mult_cb, bdiv_cb, bmul, accw, packed);
    uint8_t* const dst = static_cast<uint8_t*>(a.y) + off;
    if (cb + kLaneCh <= a.OC)
      runs_store<NT>(dst, packed, through);
    else
      runs_store_some<NT>(dst, packed, a.OC - cb);
  }
}

template <int MODE, int POST, int NT, bool PLAIN = false>
__global__ __launch_bounds__(kCrThreads, 3) void conv_runs_kernel(ConvRunArgs a) {
  constexpr int kCrBN = 16 * NT;  // output channels per block (grid y)
  constexpr int kLaneCh = 4 * NT; // consecutive channels of one pixel in a lane
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ __attribute__((aligned(16))) int s_acc0[kCrBN];
  __shared__ __attribute__((aligned(16))) float s_mult[kCrBN];
  __shared__ __attribute__((aligned(16))) float s_bdiv[kCrBN];

  const int t = threadIdx.x, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int pj = lane & 15, pq = lane >> 4;
  const int n0 = static_cast<int>(blockIdx.y) * kCrBN;
  const int KS = a.KS;
  uint8_t* const sX = lds;                  // staged image rows

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
  // the weight operands of this block's 64 channels, laid out per lane at prepack
  v4i wreg[NT][kCrMaxKS];
  {
    const uint8_t* const wsrc = a.w_runs + (static_cast<int64_t>(blockIdx.y) * NT * KS * kWave + lane) * 16;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int ks = 0; ks < kCrMaxKS; ++ks)
        wreg[nt][ks] = ks < KS ? ld16(wsrc + (nt * KS + ks) * (kWave * 16)) : v4i{0, 0, 0, 0};
  }
  __syncthreads();
  // this lane's piece of every k-step: staged row and byte inside the run
  int lk[kCrMaxKS];  // (a multiple of 16) | the row's share of the alignment shift, (kh * (row bytes % 16)) % 16
#pragma unroll
  for (int ks = 0; ks < kCrMaxKS; ++ks) {
    const int koff = ks * 64 + pq * 16;
    int kh = koff / a.RP, ro = koff - kh * a.RP;
    if (kh >= a.KH) {  // past the last kernel row: zero weights, any staged bytes
      kh = a.KH - 1;
      ro = 0;
    }
    lk[ks] = (kh * a.pitch + ro) | ((kh * (a.W * a.IC)) & 15);
  }
  float bmul = 1.0f;
  if constexpr (MODE != kOutAcc32) bmul = bias_mul(a.w_scale_stride == 0, a.x_scale * a.w_scales[0]);

  const int row_bytes = a.W * a.IC;
  const int tile_mt = a.TR * a.mtw;
  // The staged rows of a tile pass through registers, requested one tile ahead, so that they
  // arrive while the tile in hand is multiplied.  The unit of the copy is 1 KB of one staged
  // row, one 16-byte load per lane; unit u belongs to wave u % 4 (the host sizes the tiles
  // for at most kCrUnits units per wave).  Staged row r starts
  //   shift(r) = (c0 + r * (row bytes % 16)) % 16
  // bytes before the tile's first byte of that image row, so that every load is an aligned
  // 16 bytes of memory: LDS byte q of the row is image-row byte iwb0 - shift(r) + q.
  const int segs = (a.pitch + 1023) >> 10, units = a.rows_in * segs;
  v4i pre[kCrUnits];
  struct TilePos {
    int b, oh0, ow0, c0;
    int ih0, iwb0;        // image row and byte in the row of the tile's first staged byte (before the shift)
    int64_t first;        // the same as a byte offset into the tensor
    int edge;             // some load may reach outside the tensor
  };
  const int rb15 = row_bytes & 15;
  const int64_t x_bytes = static_cast<int64_t>(a.B) * a.H * row_bytes;
  auto tile_pos = [&](uint32_t tile) {
    TilePos tp;
    const uint32_t trb = tile / static_cast<uint32_t>(a.tiles_w);
    const int tcol = static_cast<int>(tile - trb * static_cast<uint32_t>(a.tiles_w));
    tp.b = static_cast<int>(trb / static_cast<uint32_t>(a.tiles_h));
    const int trow = static_cast<int>(trb) - tp.b * a.tiles_h;
    tp.oh0 = trow * a.TR;
    tp.ow0 = tcol * a.TW;
    tp.ih0 = tp.oh0 * a.sh - a.ph;
    tp.iwb0 = (tp.ow0 * a.sw - a.pw) * a.IC;
    tp.first = (static_cast<int64_t>(tp.b) * a.H + tp.ih0) * row_bytes + tp.iwb0;
    tp.c0 = static_cast<int>((reinterpret_cast<uintptr_t>(a.x) + static_cast<uintptr_t>(tp.first)) & 15);
    tp.edge = tp.first < 16 || tp.first + static_cast<int64_t>(a.rows_in) * row_bytes + a.pitch + 16 > x_bytes;
    return tp;
  };
  // Unit `slot` of this wave: staged row, first LDS byte of the unit in that row (-1: none).
  auto unit_pos = [&](int slot, int* r, int* q0) {
    const int u = wave + kCrWaves * slot;
    *r = segs == 1 ? u : u / segs;
    *q0 = u < units ? (u - *r * segs) << 10 : -1;
  };
  // The loads only.  A load may hang over either end of its image row into the neighbouring
  // rows (store_tile overwrites those bytes); nothing here uses a loaded value, so nothing
  // waits.  Only in the first and the last tiles of the tensor can a load reach outside it;
  // those tiles check every byte.
  auto request = [&](const TilePos& tp) {
#pragma unroll
    for (int slot = 0; slot < kCrUnits; ++slot) {
      int r, q0;
      unit_pos(slot, &r, &q0);
      if (q0 < 0 || static_cast<unsigned>(tp.ih0 + r) >= static_cast<unsigned>(a.H)) continue;  // (wave-uniform)
      const int q = q0 + 16 * lane;
      const int64_t rel = tp.first + static_cast<int64_t>(r) * row_bytes - ((tp.c0 + r * rb15) & 15) + q0;
      if (q >= a.pitch) continue;
      if (!tp.edge) {
        pre[slot] = *reinterpret_cast<const v4i*>(a.x + rel + 16 * lane);
      } else {
        uint32_t w4[4] = {0, 0, 0, 0};
        for (int jj = 0; jj < 16; ++jj) {
          const int64_t o = rel + 16 * lane + jj;
          if (o >= 0 && o < x_bytes) w4[jj >> 2] |= static_cast<uint32_t>(a.x[o]) << (8 * (jj & 3));
        }
        pre[slot] = v4i{static_cast<int>(w4[0]), static_cast<int>(w4[1]), static_cast<int>(w4[2]), static_cast<int>(w4[3])};
      }
    }
  };
  // Into LDS with the sign flip; then the bytes outside the image -- whole rows above and
  // below it, the ends of a row left and right of it -- become the activation zero point.
  // A wave pads its own units, after its own stores to them.
  auto store_tile = [&](const TilePos& tp) {
    const int xw = static_cast<int>(a.x_xor), pw4 = static_cast<int>(a.pad_word ^ a.x_xor);
    const v4i xmask = {xw, xw, xw, xw}, padv = {pw4, pw4, pw4, pw4};
#pragma unroll
    for (int slot = 0; slot < kCrUnits; ++slot) {
      int r, q0;
      unit_pos(slot, &r, &q0);
      if (q0 < 0) continue;
      const bool row_in = static_cast<unsigned>(tp.ih0 + r) < static_cast<unsigned>(a.H);
      uint8_t* const row = sX + r * a.pitch;
      const int q = q0 + 16 * lane;
      if (q < a.pitch) *reinterpret_cast<v4i*>(row + q) = row_in ? (pre[slot] ^ xmask) : padv;
      if (!row_in) continue;
      const int shift = (tp.c0 + r * rb15) & 15;
      const int qend = q0 + 1024 < a.pitch ? q0 + 1024 : a.pitch;
      // left of the image row: LDS bytes [0, shift - iwb0); right of it: [shift + row bytes - iwb0, pitch)
      const int left = shift - tp.iwb0 < qend ? shift - tp.iwb0 : qend;
      for (int i = q0 + lane; i < left; i += kWave) row[i] = static_cast<uint8_t>(pw4);
      const int right = shift + row_bytes - tp.iwb0 > q0 ? shift + row_bytes - tp.iwb0 : q0;
      for (int i = right + lane; i < qend; i += kWave) row[i] = static_cast<uint8_t>(pw4);
    }
  };
  TilePos cur{};
  if (static_cast<int>(blockIdx.x) < a.tiles) {
    cur = tile_pos(blockIdx.x);
    request(cur);
  }
  for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    const int b = cur.b, oh0 = cur.oh0, ow0 = cur.ow0, c0 = cur.c0;
    // ---- the staged rows of this tile into LDS, the next tile's on their way
    store_tile(cur);
    __syncthreads();
    if (tile + static_cast<int>(gridDim.x) < a.tiles) {
      cur = tile_pos(static_cast<uint32_t>(tile) + gridDim.x);
      request(cur);
    }

    // ---- multiply: 16 pixels of one output row per wave and turn
    const int tw_valid = a.OW - ow0 < a.TW ? a.OW - ow0 : a.TW;
    const int th_valid = a.OH - oh0 < a.TR ? a.OH - oh0 : a.TR;
    int orow = 0, mcol = wave;  // this wave's piece: row of the tile, 16-pixel piece of the row
    for (int mt = wave; mt < tile_mt; mt += kCrWaves, mcol += kCrWaves) {
      while (mcol >= a.mtw) {
        mcol -= a.mtw;
        ++orow;
      }
      if (orow >= th_valid || mcol * 16 >= tw_valid) continue;  // (the same for the whole wave)
      const int pcol = mcol * 16 + pj;
      const int pc = pcol < tw_valid ? pcol : tw_valid - 1;
      const int base = orow * a.sh * a.pitch + pc * a.sw * a.IC;
      const int c0r = c0 + orow * a.sh * rb15;  // alignment shift of staged row orow * stride, before the % 16
      v4i acc[NT];  // start: the zero point's share, acc_coef * colsum
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = *reinterpret_cast<const v4i*>(&s_acc0[kLaneCh * pq + 4 * nt]);
#pragma unroll
      for (int ks = 0; ks < kCrMaxKS; ++ks) {
        if (ks < KS) {
          const int addr = base + (lk[ks] & ~15) + ((c0r + lk[ks]) & 15);
          const uint32_t* const src = reinterpret_cast<const uint32_t*>(sX + (addr & ~3));
          const uint32_t sb = static_cast<uint32_t>(addr & 3);
          const uint32_t d0 = src[0], d1 = src[1], d2 = src[2], d3 = src[3], d4 = src[4];
          const v4i xv = {static_cast<int>(__builtin_amdgcn_alignbyte(d1, d0, sb)),
                          static_cast<int>(__builtin_amdgcn_alignbyte(d2, d1, sb)),
                          static_cast<int>(__builtin_amdgcn_alignbyte(d3, d2, sb)),
                          static_cast<int>(__builtin_amdgcn_alignbyte(d4, d3, sb))};
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[nt][ks], xv, acc[nt], 0, 0, 0);
        }
      }
      // ---- requantise and store: this lane has channels n0 + 4 NT pq .. + 4 NT - 1 of pixel pj
      if (pcol >= tw_valid) continue;
      const int64_t opix = (static_cast<int64_t>(b) * a.OH + oh0 + orow) * a.OW + ow0 + pcol;
      const int cb = n0 + kLaneCh * pq;
      if (cb >= a.OC) continue;
      const int64_t off = opix * a.OC + cb;
      RunsResidual<NT> accw{};
      if (POST == 1 || (POST == 2 && a.post.accum != nullptr)) accw = runs_residual<NT>(a, off, cb);
      runs_requant_store<MODE, POST, NT, PLAIN>(a, acc, off, cb, &s_mult[kLaneCh * pq], &s_bdiv[kLaneCh * pq], bmul, accw,
                                                a.through != 0);
    }
    __syncthreads();  // the staged rows are overwritten by the next tile
  }
}

// Pointwise layers (1 x 1, stride 1, no padding, one group) over at most 256 input channels,
// on the same per-lane weight layout: here a pixel's IC bytes *are* the run, a lane's MFMA
// operand for pixel p and k-step ks is the 16 bytes at p * IC + 64 ks + 16 (lane / 16) of the
// input -- straight from memory, any alignment, no staging -- and what it picks up past the
// pixel's last channel (the next pixel's bytes) meets zero weights.
//
// A wave owns one channel block for the whole launch, its weights (NT x KSN operands) and the
// requantisation constants of the lane's 4 NT channels in registers, and walks every G-th 16-pixel
// piece of the image, D pieces' bytes (input and residual) on their way: a load per k-step, the MFMAs,
// eight vector instructions per value (four without a residual) and one store, no LDS and no barrier.  The waves
// of neighbouring channel blocks read the same pieces at the same time, from one L1.  With the weights and constants in
// LDS and every channel block over a piece in turn, the LDS reads were a third of its instructions and the residual a
// latency per block (64 -> 256 channels with a residual on 56 x 56 at batch 32, 58 MB: 27.9 us).
//
// A launch has a handful of pieces per wave, so what bounds it is a wave's chain: arguments, set-up, first bytes, then
// pieces whose loads, products and stores follow one another.  Hence all requests of the set-up leave together, the
// constants first and each wave's its own (the bias used to be asked for after the scales had come, and the block met
// at a barrier), the wave's place in the grid is a multiplication, not a division, and a piece that lies inside the
// tensors takes its addresses from the scalar unit and keeps an exact count of the requests on their way.  us, before |
// after: the layer above 15.2 | 13.7, 256 -> 64 on the same image (32 MB) 9.6 | 8.0, 24 -> 144 there 10.2 | 9.5 and on
// one image of 57 x 43 4.0 | 3.2, 16 -> 96 on 112 x 112 at batch 32 18.0 | 15.3, 512 channels with a residual from 128
// on 28 x 28 at batch 8 7.2 | 6.2.
// (256 -> 64 with four pieces ahead instead of two: 9.3 against 8.9 us.)
// a.tiles: the number of 16-pixel pieces.
template <int KSN>
constexpr int kCrPointwiseDepth = KSN == 1 ? 4 : 2;
constexpr int kCrXcdBlocks = 8;  // channel blocks from which on the waves of a group of pixels sit on one XCD

// THROUGH: the stores of whole lanes are st16_through / st8_through.  (As a branch in the kernel it took registers: SiLU
// behind 65 to 128 channels spilled ten instead of five and was 5 to 8 % slower, 4.2 | 4.5 us at 128 -> 192 on 37 x 38, and
// 16 to 64 channels without a residual had three waves a SIMD instead of four.)
template <int MODE, int POST, int NT, int KSN, bool PLAIN, bool THROUGH>
__global__ __launch_bounds__(kCrThreads, KSN == 4 ? 2 : 3) void conv_runs_pointwise_kernel(ConvRunArgs a) {
  constexpr int kCrBN = 16 * NT;   // output channels per channel block
  constexpr int kLaneCh = 4 * NT;  // consecutive channels of one pixel in a lane
  constexpr int D = kCrPointwiseDepth<KSN>;
  // constants of the channels of this block's waves, each wave its own
  __shared__ __attribute__((aligned(16))) int s_acc0[kCrWaves * kCrBN];
  __shared__ __attribute__((aligned(16))) float s_mult[kCrWaves * kCrBN];
  __shared__ __attribute__((aligned(16))) float s_bdiv[kCrWaves * kCrBN];
  const int t = threadIdx.x, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int pj = lane & 15, pq = lane >> 4;
  const int KS = a.KS;
  const int nblk = a.nblk, groups = a.groups;
  // With eight and more channel blocks the waves of one group of pixels sit in several blocks: on one XCD they share the
  // pixels' bytes and the output lines where two channel blocks meet (97 -> 582 channels on 22 x 38 x 81 34.9 -> 30.8 us,
  // 128 -> 768 on 11 x 17 x 48 8.4 -> 8.0; fewer share nothing and stream worse: 24 -> 144 at batch 32 9.9 -> 12.2, 128 ->
  // 273 with a residual 7.3 -> 8.0).  Where some groups, the first ones, have a piece more than the rest, the groups are
  // dealt to the XCDs in turn: in one run they kept one XCD busy for longer (96 -> 512 with SiLU on 2 x 59 x 59, 436 pieces
  // for 384 groups: 8.8 -> 7.5 us).
  const uint32_t xcd = blockIdx.x & a.xcd_mask;
  const uint32_t block = xcd * a.xcd_blocks + (xcd < a.xcd_longer ? xcd : a.xcd_longer) + (blockIdx.x >> a.xcd_shift);
  const uint32_t w = block * kCrWaves + static_cast<uint32_t>(wave);
  const int in_run = static_cast<int>(nblk == 1 ? w : __umulhi(w, a.nblk_magic));
  const int cb = static_cast<int>(w) - in_run * nblk;
  const int g = (in_run << a.deal_shift) + static_cast<int>(xcd & a.deal_mask);
  if (g >= groups || g >= a.tiles) return;  // (no barrier below: the waves share nothing)

  // Every request of the set-up leaves before anything is waited for, the constants first: with the bias behind a
  // branch of its own its latency (cold: most of a microsecond) came on top of the scales'.
  const int ci = lane % kCrBN;
  const int cn = cb * kCrBN + ci < a.OC ? cb * kCrBN + ci : 0;
  const int c_cs = a.colsum[cn];
  float c_ws = 1.f, c_b = 0.f;
  if constexpr (MODE != kOutAcc32) {
    c_ws = a.w_scales[cn * a.w_scale_stride];
    const float* const bsrc = a.bias != nullptr ? a.bias : a.w_scales;  // a load that always has an address
    c_b = bsrc[a.bias != nullptr ? cn : 0];
  }
  const int npix = a.B * a.H * a.W;
  const int64_t x_bytes = static_cast<int64_t>(npix) * a.IC;
  // A piece all of whose bytes exist (the first a.whole ones): addresses are the piece's, the same for the whole wave,
  // plus an offset of the lane that never changes, so that a piece costs no vector instruction for them.
  const bool residual = POST == 1 || (POST == 2 && a.post.accum != nullptr);
  const int cl = cb * kCrBN + kLaneCh * pq;  // this lane's first channel
  const bool all_ch = (cb + 1) * kCrBN <= a.OC;  // every lane of the wave has its 4 NT channels
  const uint32_t yo = static_cast<uint32_t>(pj * a.OC + cl);
  // (a lane at the end of the channels reads its residual bytes as the pixel's last 4 NT and shifts them down)
  const int over = cl + kLaneCh - a.OC;
  const uint32_t ro = yo - static_cast<uint32_t>(over > 0 && over < kLaneCh ? over : over > 0 ? cl : 0);
  uint32_t xo[KSN];
#pragma unroll
  for (int ks = 0; ks < KSN; ++ks) {
    const int k0 = ks * 64 + pq * 16;
    xo[ks] = static_cast<uint32_t>(pj * a.IC + (k0 < a.RP ? k0 : 0));
  }
  // Piece number i of this wave.  A number past the last asks for the first piece's first bytes instead, the same for all
  // lanes: the count of requests on their way stays exact, which one under a condition would end (the compiler then
  // waits for all of them), and it costs next to nothing.
  const int mine = g < a.whole ? (a.whole - g + groups - 1) / groups : 0;  // whole pieces of this wave
  const auto fetch = [&](int i, v4i (&xv)[KSN], RunsResidual<NT>& r) {
    const int64_t first = i < mine ? (g + i * groups) * int64_t{16} : 0;
    const uint32_t keep = i < mine ? ~0u : 0u;
    const uint8_t* const src = a.x + first * a.IC;
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks) xv[ks] = ld16_any(src + (xo[ks] & keep));
    if (!residual) return;
    const uint8_t* const rsrc = a.post.accum + first * a.OC + (ro & keep);
    if constexpr (NT == 4) {
      const v4i v = ld16_any(rsrc);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) r.w[nt] = static_cast<uint32_t>(v[nt]);
    } else {
      const v2i v = reinterpret_cast<const V2iAnyAlignment*>(rsrc)->v;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) r.w[nt] = static_cast<uint32_t>(v[nt]);
    }
  };
  // the first pieces' bytes and the weights are asked for before the constants are set up
  v4i xr[D][KSN];
  RunsResidual<NT> rr[D];
  v4i wreg[NT][KSN];
#pragma unroll
  for (int i = 0; i < D; ++i) {
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks) xr[i][ks] = v4i{0, 0, 0, 0};
    rr[i] = RunsResidual<NT>{};
  }
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < D; ++i) fetch(i, xr[i], rr[i]);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks)
      wreg[nt][ks] = ks < KS ? ld16(a.w_runs + ((static_cast<int64_t>(cb) * NT + nt) * KS + ks) * (kWave * 16) + lane * 16)
                                      : v4i{0, 0, 0, 0};
  // the wave's constants, a channel per lane (two IEEE divisions each), then to the lanes that want them
  float bmul = 1.0f;
  {
    float mult = 0.f, bdiv = 0.f;
    if constexpr (MODE != kOutAcc32) {
      const float atw = a.x_scale * c_ws;
      mult = atw / a.out_scale;
      bdiv = a.bias != nullptr ? bias_term(a.w_scale_stride == 0, c_b, atw) : 0.f;
      bmul = bias_mul(a.w_scale_stride == 0, atw);  // (per tensor: the same for every channel)
    }
    s_acc0[wave * kCrBN + ci] = a.acc_coef * c_cs;
    s_mult[wave * kCrBN + ci] = mult;
    s_bdiv[wave * kCrBN + ci] = bdiv;
    wave_sync_lds();
  }
  v4i acc0[NT];
  float mult[kLaneCh], bdiv[kLaneCh];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int at = wave * kCrBN + kLaneCh * pq + 4 * nt;
    acc0[nt] = *reinterpret_cast<const v4i*>(&s_acc0[at]);
    const v4f m = *reinterpret_cast<const v4f*>(&s_mult[at]), b = *reinterpret_cast<const v4f*>(&s_bdiv[at]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      mult[4 * nt + r] = m[r];
      bdiv[4 * nt + r] = b[r];
    }
  }
  const int flip_word = static_cast<int>(a.x_xor);
  const v4i flip = {flip_word, flip_word, flip_word, flip_word};
  const auto multiply = [&](const v4i (&xv)[KSN], v4i (&acc)[NT]) {
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks) {
      const v4i xf = xv[ks] ^ flip;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[nt][ks], xf, ks == 0 ? acc0[nt] : acc[nt], 0, 0, 0);
    }
  };
  const auto whole_piece = [&](int i, int n, auto all_ch_tag) {
    v4i acc[NT];
    multiply(xr[i], acc);
    RunsResidual<NT> accw = rr[i];
    fetch(n + D, xr[i], rr[i]);
    const int64_t base = static_cast<int64_t>(g + n * groups) * (16 * a.OC);
    if constexpr (MODE == kOutAcc32) {
      if (cl < a.OC) runs_requant_store<MODE, POST, NT, PLAIN>(a, acc, base + yo, cl, mult, bdiv, bmul, accw, false);
    } else {
      uint32_t packed[NT];
      uint8_t* const dst = static_cast<uint8_t*>(a.y) + base;
      if constexpr (decltype(all_ch_tag)::value) {
        runs_requant<MODE, POST, NT, PLAIN>(a, acc, mult, bdiv, bmul, accw, packed);
        runs_store<NT>(dst + yo, packed, THROUGH);
      } else {
        if (residual && over > 0 && over < kLaneCh) {
          v4i v = {0, 0, 0, 0};
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) v[nt] = static_cast<int>(accw.w[nt]);
          v = shift_down_bytes(v, over);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) accw.w[nt] = static_cast<uint32_t>(v[nt]);
        }
        runs_requant<MODE, POST, NT, PLAIN>(a, acc, mult, bdiv, bmul, accw, packed);
        if (over <= 0)
          runs_store<NT>(dst + yo, packed, THROUGH);
        else if (over < kLaneCh)
          runs_store_some<NT>(dst + yo, packed, kLaneCh - over);
      }
    }
  };
  // (one copy of the D pieces, left at any of them: waves with a piece or two would pay for fetching a second one)
  const auto walk = [&](auto all_ch_tag) {
    for (int n = 0;; n += D) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        if (n + i >= mine) return;
        whole_piece(i, n + i, all_ch_tag);
      }
    }
  };
  if (MODE != kOutAcc32 && all_ch)
    walk(std::true_type{});
  else
    walk(std::false_type{});
  // what is left at the tensor's end (one piece or two of the launch): every address checked
  for (int piece = g + mine * groups; piece < a.tiles; piece += groups) {
    const int pix = piece * 16 + pj < npix ? piece * 16 + pj : npix - 1;
    const int64_t row = static_cast<int64_t>(pix) * a.IC;
    v4i xv[KSN], acc[NT];
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks) {
      // (a pixel or bytes that do not exist: any others -- nothing of them is stored, or their weights are zero)
      const int k0 = ks * 64 + pq * 16;
      const TailRead r = tail_read16(row + (k0 < a.RP ? k0 : 0), x_bytes);  // (the host: a tensor of at least 16 bytes)
      xv[ks] = ld16_any(a.x + r.at);
      if (r.shift > 0) xv[ks] = shift_down_bytes(xv[ks], r.shift);  // the tensor's last few bytes
    }
    multiply(xv, acc);
    if (piece * 16 + pj < npix && cl < a.OC) {
      const int64_t off = static_cast<int64_t>(pix) * a.OC + cl;
      RunsResidual<NT> accw{};
      if (residual) accw = runs_residual<NT>(a, off, cl);
      runs_requant_store<MODE, POST, NT, PLAIN>(a, acc, off, cl, mult, bdiv, bmul, accw, THROUGH);
    }
  }
}

}  // namespace tmq
