// quantized::conv2d for gfx950: NHWC implicit GEMM on the int8 MFMA core.
//
// GEMM view per group: rows m = (b, oh, ow) output pixels, columns n = output
// channels of the group, k = (kh, kw, ic) with every tap padded to a multiple
// of 16 input channels, so one 16-byte k-chunk is one run of 16 channels of one
// input pixel -- a single aligned load from the NHWC activation tensor.
// Taps outside the image are filled with the activation zero point (real value
// 0), which the accumulator start value then cancels exactly.
#include <atomic>
#include <type_traits>

#include "conv_image.h"
#include "gemm_i8_wloop.h"
#include "conv_runs.h"
#include "conv_depthwise.h"
#include "conv_tile.h"
#include "gemm_i8_core.h"

static_assert(sizeof(tmq_conv2d_geom) == 112, "tmq_conv2d_geom layout changed");
static_assert(sizeof(tmq_conv2d_desc) == 224, "tmq_conv2d_desc layout changed");
static_assert(sizeof(tmq_conv2d_post) == 24, "tmq_conv2d_post layout changed");

namespace tmq {
namespace {

constexpr int64_t kKPad = 128;
constexpr int64_t kCuLds = 160 * 1024;            // LDS of a CU, what blocks that run on it at once share
constexpr int64_t kPatchRowsMinK = 2048;         // K from which on a layer may run on its patch rows (workspace) ...
constexpr int64_t kPatchRowsMaxK = 4096;         // ... and up to which it may at more pixels (patch_rows_max)
inline int64_t packed_kchunks(int64_t K) { return (K + kKPad - 1) / kKPad * (kKPad / 16); }

struct ConvShape {
  int64_t B, H, W, IC, OC, KH, KW, OH, OW;
  int64_t sh, sw, ph, pw, dh, dw, groups;
  int64_t ICg, OCg, ICgp, Kp, KC, group_bytes;
  int64_t ICgo, OCgo;  // channels per group as the caller states them (see make_shape)
  // the second weight layout, behind the first, for the kernel of conv_runs.h: k-steps
  // (0: the shape is not that kernel's), run bytes, padded run bytes, offset and size in bytes
  int64_t runs_KS, runs_RL, runs_RP, runs_off, runs_bytes;
  bool pixels4;  // ... laid out for the kernel of conv_image.h, three channels as four-byte pixels
  // depthwise layers over a multiple of 4 or at least 16 channels: a [channel][kernel row][taps padded to a multiple
  // of 4] copy of the weight for the kernel of conv_depthwise.h in the same place (0: not such a layer)
  int64_t taps_bytes;
};

int make_shape(const tmq_conv2d_geom* g, ConvShape* s) {
  if (g == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (g->B < 0 || g->H <= 0 || g->W <= 0 || g->IC <= 0 || g->OC <= 0 || g->KH <= 0 || g->KW <= 0 ||
      g->stride_h <= 0 || g->stride_w <= 0 || g->pad_h < 0 || g->pad_w < 0 || g->dil_h <= 0 ||
      g->dil_w <= 0 || g->groups <= 0)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (g->IC % g->groups != 0 || g->OC % g->groups != 0) return TMQ_ERR_INVALID_ARGUMENT;
  s->B = g->B; s->H = g->H; s->W = g->W; s->IC = g->IC; s->OC = g->OC; s->KH = g->KH; s->KW = g->KW;
  s->sh = g->stride_h; s->sw = g->stride_w; s->ph = g->pad_h; s->pw = g->pad_w;
  s->dh = g->dil_h; s->dw = g->dil_w; s->groups = g->groups;
  s->OH = (g->H + 2 * g->pad_h - g->dil_h * (g->KH - 1) - 1) / g->stride_h + 1;
  s->OW = (g->W + 2 * g->pad_w - g->dil_w * (g->KW - 1) - 1) / g->stride_w + 1;
  if (s->OH <= 0 || s->OW <= 0) return TMQ_ERR_INVALID_ARGUMENT;
  // Groups whose input channels are no multiple of 16 (depthwise and other narrow groups)
  // are merged: `merge` neighbouring groups become one group with a block-diagonal weight --
  // zeros where an output channel meets another group's input channels -- so that a 16-byte
  // k-chunk is again 16 channels of one pixel and the MFMA kernels take the problem.  The
  // matrix pipe multiplies the zeros at no cost that matters: these layers move bytes.
  // The merged group has as many channels as a tile of the kernels is wide (64) where the
  // group count allows.  groups / ICg / OCg below are the merged ones; the packed weight
  // is laid out for them.
  s->ICgo = g->IC / g->groups;
  s->OCgo = g->OC / g->groups;
  int64_t merge = 1;
  if (g->groups > 1 && s->ICgo % 16 != 0) {
    const int64_t low = s->ICgo & -s->ICgo;             // largest power of two in ICgo
    const int64_t v0 = 16 / (low < 16 ? low : 16);      // fewest groups that make a multiple of 16
    for (int64_t v = v0; v <= g->groups; v += v0) {
      if (v > v0 && (v * s->OCgo > 64 || v * s->ICgo > 64)) break;
      if (g->groups % v == 0) merge = v;
    }
    if ((merge * s->ICgo) % 16 != 0) merge = 1;         // (no such divisor of the group count)
  }
  s->groups = g->groups / merge;
  s->ICg = merge * s->ICgo;
  s->OCg = merge * s->OCgo;
  s->ICgp = round_up(s->ICg, 16);
  s->Kp = g->KH * g->KW * s->ICgp;
  s->KC = packed_kchunks(s->Kp);
  s->group_bytes = ceil_div(s->OCg, 16) * s->KC * 256;
  s->runs_KS = s->runs_RL = s->runs_RP = s->runs_bytes = 0;
  s->pixels4 = false;
  s->runs_off = s->groups * s->group_bytes;
  if (g->groups == 1 && g->dil_h == 1 && g->dil_w == 1) {
    s->pixels4 = g->IC == 3 && g->KH * round_up(g->KW * 4, 16) <= 64 * kCrMaxKS && !(g->KH == 1 && g->KW == 1);
    const int64_t RL = g->KW * (s->pixels4 ? 4 : g->IC), RP = round_up(RL, 16);
    if (g->KH * RP <= 64 * kCrMaxKS) {
      s->runs_RL = RL;
      s->runs_RP = RP;
      s->runs_KS = ceil_div(g->KH * RP, 64);
      const int64_t tiles = conv_runs_tiles(g->OC);  // 16-channel tiles per block
      s->runs_bytes = ceil_div(g->OC, 16 * tiles) * tiles * s->runs_KS * kWave * 16;
    }
  }
  s->taps_bytes = 0;
  if (g->groups > 1 && g->groups == g->IC && g->IC == g->OC && (g->IC % 4 == 0 || g->IC >= 16))
    s->taps_bytes = round_up(g->IC * g->KH * round_up(g->KW, 4), 16);
  // 32-bit index arithmetic inside the kernels
  if (g->H > (1 << 24) || g->W > (1 << 24) || g->IC > (1 << 24) || s->Kp > (1 << 30) ||
      g->B * s->OH * s->OW > 0x7fffffff || g->H * g->W * g->IC > 0x3fffffff)
    return TMQ_ERR_UNSUPPORTED;
  return TMQ_OK;
}

// One thread per 16-byte packed chunk (group, nb, kc, r).
__global__ __launch_bounds__(256) void conv_prepack_kernel(const int8_t* __restrict__ w,
                                                           ConvShape s, int64_t total,
                                                           uint8_t* __restrict__ packed) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  const int64_t per_group = s.group_bytes / 16;
  const int64_t g = id / per_group, lid = id % per_group;
  const int r = static_cast<int>(lid & 15);
  const int64_t kc = (lid >> 4) % s.KC, nb = (lid >> 4) / s.KC;
  const int64_t n = nb * 16 + r;
  const int64_t k0 = kc * 16;
  const int64_t tap = k0 / s.ICgp, ic0 = k0 % s.ICgp;
  uint32_t words[4] = {0, 0, 0, 0};
  if (n < s.OCg && tap < s.KH * s.KW) {
    // the output channel's own group inside a merged one: its input channels lo .. lo + ICgo - 1
    const int64_t lo = n / s.OCgo * s.ICgo;
    const int8_t* src = w + ((g * s.OCg + n) * s.KH * s.KW + tap) * s.ICgo;
    for (int b = 0; b < 16; ++b)
      if (ic0 + b >= lo && ic0 + b < lo + s.ICgo)
        words[b >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(src[ic0 + b - lo])) << (8 * (b & 3));
  }
  *reinterpret_cast<v4i*>(packed + id * 16) =
      v4i{static_cast<int>(words[0]), static_cast<int>(words[1]), static_cast<int>(words[2]),
          static_cast<int>(words[3])};
}

// One thread per 16-byte slot of the per-lane layout of conv_runs.h.
__global__ __launch_bounds__(256) void conv_prepack_runs_kernel(const int8_t* __restrict__ w, ConvShape s,
                                                                int64_t total, uint8_t* __restrict__ dst) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  *reinterpret_cast<v4i*>(dst + id * 16) =
      s.pixels4 ? conv_image_slot(w, id, static_cast<int>(s.OC), static_cast<int>(s.KH), static_cast<int>(s.KW),
                                  static_cast<int>(s.runs_RP), static_cast<int>(s.runs_KS))
                : conv_runs_slot(w, id, static_cast<int>(s.OC), static_cast<int>(s.KH), static_cast<int>(s.runs_RL),
                     static_cast<int>(s.runs_RP), static_cast<int>(s.runs_KS));
}

// One thread per byte of the [channel][kernel row][padded taps] layout of conv_depthwise.h (the
// caller's weight is [channel][kernel row][tap]).
__global__ __launch_bounds__(256) void conv_prepack_taps_kernel(const int8_t* __restrict__ w, int64_t C, int64_t KH,
                                                                int64_t KW, int64_t total, uint8_t* __restrict__ dst) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  const int64_t kwp = (KW + 3) / 4 * 4;
  const int64_t kw = id % kwp, kh = id / kwp % KH, c = id / (kwp * KH);
  dst[id] = c < C && kw < KW ? static_cast<uint8_t>(w[(c * KH + kh) * KW + kw]) : uint8_t{0};
}

__global__ __launch_bounds__(256) void conv_colsum_kernel(const int8_t* __restrict__ w, int64_t OC,
                                                          int64_t K, int32_t* __restrict__ colsum) {
  const int lane = threadIdx.x % kWave;
  const int64_t n = static_cast<int64_t>(blockIdx.x) * (256 / kWave) + threadIdx.x / kWave;
  if (n >= OC) return;
  int s = 0;
  for (int64_t i = lane; i < K; i += kWave) s += w[n * K + i];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
  if (lane == 0) colsum[n] = s;
}

// Whether the implicit GEMM has the layer's k order in a table (XConvTable); the rest walks it (XConv): kernels of 8 x 8 and
// more, K that ends before the copies' ring of three stages is full, and images of which a tile's 128 rows reach past the
// 32 bits of its offsets.
bool conv_table_takes(const ConvShape& s) {
  return s.KH * s.KW <= kConvMaxTaps && s.Kp / 16 <= kConvMaxChunks && s.Kp > 2 * kBK &&
         (128 / (s.OH * s.OW) + 2) * s.H * s.W * s.IC < (int64_t{1} << 31);
}

// Patch rows (im2col) of a convolution over whole 16-channel blocks, one group: row m = output
// pixel (b, oh, ow), k = (kh, kw, ic) as in the packed weight; one thread per 16-byte chunk.
// Taps outside the image are the activation zero point.
__global__ __launch_bounds__(256) void conv_patch_rows_kernel(const uint8_t* __restrict__ x, ConvShape s, int64_t total,
                                                              uint32_t pad_word, uint8_t* __restrict__ rows) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  const uint32_t kc = static_cast<uint32_t>(s.Kp / 16), icb = static_cast<uint32_t>(s.IC / 16);
  const uint32_t m = static_cast<uint32_t>(id / kc), c = static_cast<uint32_t>(id - static_cast<int64_t>(m) * kc);
  const uint32_t tap = c / icb, blk = c - tap * icb;
  const uint32_t kh = tap / static_cast<uint32_t>(s.KW), kw = tap - kh * static_cast<uint32_t>(s.KW);
  const uint32_t ow = m % static_cast<uint32_t>(s.OW), t = m / static_cast<uint32_t>(s.OW);
  const uint32_t oh = t % static_cast<uint32_t>(s.OH), b = t / static_cast<uint32_t>(s.OH);
  const int ih = static_cast<int>(oh * s.sh) - static_cast<int>(s.ph) + static_cast<int>(kh * s.dh);
  const int iw = static_cast<int>(ow * s.sw) - static_cast<int>(s.pw) + static_cast<int>(kw * s.dw);
  const int pw = static_cast<int>(pad_word);
  v4i v = {pw, pw, pw, pw};
  if (static_cast<unsigned>(ih) < static_cast<unsigned>(s.H) && static_cast<unsigned>(iw) < static_cast<unsigned>(s.W))
    v = ld16(x + ((static_cast<int64_t>(b) * s.H + ih) * s.W + iw) * s.IC + blk * 16);
  *reinterpret_cast<v4i*>(rows + id * 16) = v;
}

// Output pixels up to which a layer's patch rows are ahead of the implicit GEMM (run_conv has the figures).
int64_t patch_rows_max(const ConvShape& s) {
  const bool short_k = s.Kp <= kPatchRowsMaxK;
  return conv_table_takes(s) ? (short_k ? 512 : 64) : (short_k ? 1024 : 512);
}

// Whether a layer may run on its patch rows, and the bytes they take: one group over whole
// 16-channel blocks, few output pixels, a long K, and no halo tiles for it.
int64_t patch_rows_bytes(const tmq_conv2d_geom& g, const ConvShape& s, bool pinned) {
  if (g.groups != 1 || s.IC % 16 != 0) return 0;
  const int64_t rows = s.B * s.OH * s.OW;
  if (rows == 0 || rows * (s.Kp / 16) > 0x7fffffff) return 0;
  if (!pinned) {
    const bool pointwise = s.KH == 1 && s.KW == 1 && s.ph == 0 && s.pw == 0;
    if (pointwise && s.sh == 1 && s.sw == 1) return 0;  // (already rows)
    if (pointwise) {
      // A pointwise layer with a stride: its patch rows are the pixels it reads, gathered.  From 512 input
      // channels on (batch 32: 512 -> 1024 on 28 x 28 19.5 -> 13.1 us, 1024 -> 2048 on 14 x 14 16.9 -> 12.8 us; batch 8,
      // 1024 -> 2048: 9.9 -> 8.8 us; 256 -> 512 on 56 x 56 level at batch 32 and behind at batch 8, 8.8 against 9.4 us).
      // (eight images, 512 -> 1024 on 28 x 28: 9.0 against 7.9 us on the implicit GEMM)
      if (s.IC < 512 || rows * s.IC * s.OC < (s.IC >= 1024 ? 500000000 : 2000000000)) return 0;
    } else if (rows > patch_rows_max(s) || s.Kp < kPatchRowsMinK) {
      return 0;
    }
  }
  return rows * s.Kp;
}

// One group whose channel count is no multiple of 16 and whose kernel rows are too long for the
// byte-run kernel (3 x 3 over 40 channels, 11 x 11 over 3): with scratch memory the input is
// copied once with every pixel's channels padded to whole 16-channel blocks, and the MFMA kernels
// run on the copy -- the packed weight already holds zeros at the padded positions of K, so what
// the padding bytes are does not matter.  The bytes of that copy, 0 when the layer is not such a one.
int64_t padded_input_bytes(const tmq_conv2d_geom& g, const ConvShape& s, bool pinned) {
  if (g.groups != 1 || s.IC % 16 == 0) return 0;
  if (!pinned && s.runs_KS != 0) return 0;
  const int64_t pixels = s.B * s.H * s.W, blocks = ceil_div(s.IC, 16);
  if (pixels * s.IC < 16 || pixels * blocks > 0x7fffffff) return 0;
  return pixels * blocks * 16;
}

// kPadBlocks 16-byte blocks of the padded copy per thread, each read as 16 bytes wherever they lie (the last block of a
// pixel runs on into the next pixel's bytes; the tensor's last ones are read from its last 16 bytes).  Bound by memory:
// 582 channels on 22 x 38 x 81, 39 MB in and 40 out, 41.8 us with sixteen byte loads per block and a 64-bit division, 11.8 so.
constexpr int kPadBlocks = 4;
__global__ __launch_bounds__(256) void conv_pad_channels_kernel(const uint8_t* __restrict__ x, int IC, int blocks,
                                                                uint32_t total, int64_t bytes, uint8_t* __restrict__ dst) {
  const uint32_t id0 = blockIdx.x * (256u * kPadBlocks) + threadIdx.x;
  v4i v[kPadBlocks];
  int past[kPadBlocks];  // bytes a block was read too early
#pragma unroll
  for (int u = 0; u < kPadBlocks; ++u) {
    const uint32_t id = id0 + u * 256u < total ? id0 + u * 256u : total - 1;
    const uint32_t pixel = id / static_cast<uint32_t>(blocks);
    const int64_t off = static_cast<int64_t>(pixel) * IC + (id - pixel * static_cast<uint32_t>(blocks)) * 16;
    const int64_t at = off + 16 <= bytes ? off : bytes - 16;
    past[u] = static_cast<int>(off - at);
    v[u] = ld16_any(x + at);
  }
#pragma unroll
  for (int u = 0; u < kPadBlocks; ++u) {
    const uint32_t id = id0 + u * 256u;
    if (id < total) *reinterpret_cast<v4i*>(dst + static_cast<int64_t>(id) * 16) = past[u] > 0 ? shift_down_bytes(v[u], past[u]) : v[u];
  }
}

struct PlainArgs {
  const uint8_t* x;
  const uint8_t* w_packed;
  const int32_t* colsum;
  const float* w_scales;
  const float* bias;
  int32_t w_scale_stride, x_signed, x_zp;
  float x_scale, out_scale, zp_f, lo_f, hi_f;
  void* y;
  PostOps post;
};

// Direct convolution, one thread per output value: any channel count, any
// grouping, any alignment.  Accumulates (x - x_zp) * w over in-image taps.
template <int MODE>
__global__ __launch_bounds__(256) void conv_plain_kernel(ConvShape s, PlainArgs a) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t rows = s.B * s.OH * s.OW;
  if (id >= rows * s.OC) return;
  const int64_t oc = id % s.OC, m = id / s.OC;
  const int64_t g = oc / s.OCg, n = oc % s.OCg;
  const int64_t ow = m % s.OW, oh = (m / s.OW) % s.OH, b = m / (s.OW * s.OH);
  const uint8_t* wp = a.w_packed + g * s.group_bytes;
  const int64_t sub = n / s.OCgo * s.ICgo;  // first input channel of the channel's own group inside a merged one
  int acc = 0;
  for (int64_t kh = 0; kh < s.KH; ++kh) {
    const int64_t ih = oh * s.sh - s.ph + kh * s.dh;
    if (ih < 0 || ih >= s.H) continue;
    for (int64_t kw = 0; kw < s.KW; ++kw) {
      const int64_t iw = ow * s.sw - s.pw + kw * s.dw;
      if (iw < 0 || iw >= s.W) continue;
      const uint8_t* xp = a.x + ((b * s.H + ih) * s.W + iw) * s.IC + g * s.ICg + sub;
      const int64_t kbase = (kh * s.KW + kw) * s.ICgp + sub;
      for (int64_t ic = 0; ic < s.ICgo; ++ic) {
        const int xv = a.x_signed ? static_cast<int>(static_cast<int8_t>(xp[ic])) : static_cast<int>(xp[ic]);
        const int64_t k = kbase + ic;
        const int wv = static_cast<int8_t>(wp[(((n >> 4) * s.KC + (k >> 4)) * 16 + (n & 15)) * 16 + (k & 15)]);
        acc += (xv - a.x_zp) * wv;
      }
    }
  }
  if (MODE == kOutAcc32) {
    static_cast<int32_t*>(a.y)[id] = acc;
  } else {
    const float atw = a.x_scale * a.w_scales[oc * a.w_scale_stride];
    const float mult = atw / a.out_scale;
    float v = static_cast<float>(acc);
    if (a.bias != nullptr)
      v = __builtin_fmaf(bias_term(a.w_scale_stride == 0, a.bias[oc], atw), bias_mul(a.w_scale_stride == 0, atw), v);
    float ab = v * mult;
    if (a.post.accum != nullptr) {
      const uint8_t b8 = a.post.accum[id];
      const int qa = a.post.accum_signed ? static_cast<int>(static_cast<int8_t>(b8)) : static_cast<int>(b8);
      const float ad = static_cast<float>(qa - a.post.accum_zp) * a.post.amult;
      ab = ab + ad;
    }
    if (a.post.silu) ab = silu_in_output_units(ab, a.post.silu_c, a.post.silu_c_tail);
    float r = __builtin_rintf(ab) + a.zp_f;
    r = __builtin_amdgcn_fmed3f(r, a.lo_f, a.hi_f);
    static_cast<uint8_t*>(a.y)[id] = static_cast<uint8_t>(static_cast<int>(r));
  }
}

template <int BM, int BN, int WM, int WN, int MODE, bool DMA, int KW = 1, bool THROUGH = true, class XSRC>
int launch_conv_gemm(const GemmArgs& a, const XSRC& xs, hipStream_t s) {
  const int64_t blocks = ceil_div(a.M, BM) * ceil_div(a.N, BN);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  uint32_t lds = 0;
  if constexpr (std::is_same<XSRC, XConvTable>::value) lds = conv_table_bytes(xs.chunks);
  enqueue(gemm_i8_kernel<BM, BN, WM, WN, MODE, XSRC, DMA ? 3 : 4, DMA, KW, false, THROUGH>,
          dim3(static_cast<unsigned>(blocks)), dim3(WM * WN * KW * kWave), lds, s, a, xs);
  return launch_status();
}
// Tiles that are chosen for outputs of any size (several wave groups: up to 256 and 512 tiles).
template <int BM, int BN, int WM, int WN, int MODE, bool DMA, class XSRC>
int launch_conv_gemm_any_size(const GemmArgs& a, const XSRC& xs, hipStream_t s) {
  if constexpr (MODE != kOutAcc32) {
    if (!bytes_through(a)) return launch_conv_gemm<BM, BN, WM, WN, MODE, DMA, 1, false>(a, xs, s);
  }
  return launch_conv_gemm<BM, BN, WM, WN, MODE, DMA>(a, xs, s);
}

// Tiles of the implicit GEMM.  kConvGroups2/4, kConvTall2: k-split wave groups, register staging (64 x 64 and 128 x 64).
enum ConvGemmTile { kConv64, kConvGroups2, kConvGroups4, kConvTall2, kConvRows256, kConv128, kConv256 };

// The one expected to end first, by times measured on 3 x 3 layers over 176 .. 4096 channels, 5 x 5 and 7 x 7 ones over up
// to 1024, and 49 .. 40960 pixels (us; u = tiles / 256 CUs, st = stages of 64 k-bytes):
//   64 x 64      4.0 + 0.25 u + st max(0.19 up to one tile per CU or else 0.24, 0.08 + 0.112 u)
//   128 x 64, two wave groups: 5.5 + 0.195 st for up to 256 tiles and K from 32 stages on
//   128 x 128    1.3, for each full round of the chip (three blocks on a CU, two or one where the table's LDS leaves no room
//                for more) 5.0 + 0.8, 0.55 or 0.28 st, for the last one 5.0 + st (0.28 for u <= 1, 0.35 + 0.1 u for u <= 2,
//                0.3 + 0.19 u for u <= 3)
//   128 x 256    1.0, for each full round (two blocks on a CU or one) 5.0 + 0.9 or 0.44 st, for the last one
//                5.0 + st (0.36 + 0.08 u for u <= 1, 0.52 + 0.23 u for u <= 2)
//                (a residual or SiLU in the epilogue costs the lone block of a big tile 2 and 3.5 more)
// and by tile count alone, up to 256 tiles of 64 x 64: four wave groups from 128 stages on (1024 -> 1024 on 14 x 14 23.7 with
// two, 22.3 with four; K = 9216, 176 tiles 23.7, 23.3), two from 32 on.  The groups' runs may differ by a stage (147 stages,
// 56 tiles: one group 33.2, two 24.5, four 24.0).
// What the rule changed, from 64 x 64 by fewer than 16384 pixels and 128 x 128 beyond: 512 -> 512 on 9 x 33 x 30 47 -> 34,
// on 16 x 28 x 28 62 -> 36, on 32 x 28 x 28 88 -> 67 (128 x 256); 384 -> 384 on 9 x 33 x 30 29 -> 22 (128 x 128).  On 90 random
// layers with K from 10800 to 37632 and 49 to 18424 pixels it took the fastest of the six tiles each time, on 70 with an odd
// stage count from 25 to 147 it was 1.5 % behind that one on average and 9 % at most (25 stages, where two groups are ahead).
ConvGemmTile conv_gemm_tile(int64_t M, int64_t N, int64_t stages, bool post) {
  const auto tiles = [&](int64_t bm, int64_t bn) { return ceil_div(M, bm) * ceil_div(N, bn); };
  const double st = static_cast<double>(stages), cus = 256.0;
  const int64_t t64 = tiles(64, 64);
  if (stages >= 32 && t64 <= 256) return stages >= 128 ? kConvGroups4 : kConvGroups2;
  const double u64 = t64 / cus;
  double best = 4.0 + 0.25 * u64 + st * std::max(t64 <= 256 ? 0.19 : 0.24, 0.08 + 0.112 * u64);
  ConvGemmTile tile = kConv64;
  const auto offer = [&](ConvGemmTile t, double us) {
    if (us < best) {
      best = us;
      tile = t;
    }
  };
  if (stages >= 32 && tiles(128, 64) <= 256) offer(kConvTall2, 5.5 + 0.195 * st);
  // blocks of a direct-copy tile on a CU: three stages, the channels' constants and the table
  const auto fit = [&](int64_t rows, int64_t cols, int64_t most) {
    const int64_t lds = 3 * kBK * (rows + cols) + 12 * cols + conv_table_bytes(static_cast<int>(stages * kChunks));
    return std::max<int64_t>(1, std::min(most, kCuLds / lds));
  };
  {
    const int64_t n = fit(128, 128, 3), t = tiles(128, 128), last = t % (256 * n);
    const double u = last / cus;
    const double full = n == 3 ? 0.8 : n == 2 ? 0.55 : 0.28;
    const double rate = u <= 1.0 ? 0.28 : u <= 2.0 ? 0.35 + 0.1 * u : 0.3 + 0.19 * u;
    offer(kConv128, 1.3 + (post ? 2.0 : 0.0) + t / (256 * n) * (5.0 + full * st) + (last == 0 ? 0.0 : 5.0 + rate * st));
  }
  {
    const int64_t n = fit(128, 256, 2), t = tiles(128, 256), last = t % (256 * n);
    const double u = last / cus;
    const double full = n == 2 ? 0.9 : 0.44;
    const double rate = u <= 1.0 ? 0.36 + 0.08 * u : 0.52 + 0.23 * u;
    offer(kConv256, 1.0 + (post ? 3.5 : 0.0) + t / (256 * n) * (5.0 + full * st) + (last == 0 ? 0.0 : 5.0 + rate * st));
  }
  return tile;
}

// Pointwise layers over more than 256 channels: halo tiles or this kernel, by the rounds that the former's blocks take (one
// block on a CU next to such a weight slice, so a second round is the whole chain again).  Halo time over this kernel's,
// 240 random layers from 272 to 2048 channels, geometric mean (least .. most):
//   residual alone           one round 0.89 (0.80 .. 0.95); two and three 1.21 (1.01 .. 1.45) from 384 channels on, 0.96
//                            (0.81 .. 1.21) below, where four are level (1.01, 1.03) and more 1.36
//   residual and SiLU        one round 0.97 (0.90 .. 1.06), more 1.38 (1.22 .. 1.58)
//   SiLU                     two rounds 1.49 (1.35 .. 1.61); one: up to 150 million products 1.00 (0.95 .. 1.06), beyond 1.02
//                            (0.93 .. 1.18; 1.09 from a billion on)
bool pointwise_gemm_first(const ConvShape& s, const PostOps& po, int64_t halo_rounds) {
  if (s.KH != 1 || s.KW != 1 || s.groups != 1 || s.IC <= 256) return false;
  if (po.silu && po.accum == nullptr && s.B * s.OH * s.OW * s.IC * s.OC >= 150000000) return true;
  return halo_rounds > (po.silu || s.IC >= 384 ? 1 : 4);
}

template <int MODE>
int launch_conv_gemm_tile(ConvGemmTile tile, const GemmArgs& a, const XConvTable& xs, hipStream_t s) {
  switch (tile) {
    case kConv64: return launch_conv_gemm_any_size<64, 64, 2, 2, MODE, true>(a, xs, s);
    case kConvGroups2: return launch_conv_gemm<64, 64, 2, 2, MODE, false, 2>(a, xs, s);
    case kConvGroups4: return launch_conv_gemm<64, 64, 2, 2, MODE, false, 4>(a, xs, s);
    case kConvTall2: return launch_conv_gemm<128, 64, 2, 2, MODE, false, 2>(a, xs, s);
    case kConv128: return launch_conv_gemm_any_size<128, 128, 2, 2, MODE, true>(a, xs, s);
    case kConv256: return launch_conv_gemm_any_size<128, 256, 2, 4, MODE, true>(a, xs, s);
    case kConvRows256: break;
  }
  return TMQ_ERR_UNSUPPORTED;
}

// Tiles of the layers that walk (conv_table_takes).  Up to 256 tiles of 64 x 64 four wave groups (us, one group | two |
// four: 8 x 8 over 256 channels, N = 256, 196 pixels 82 | 48 | 42, 3136 pixels 84 | 51 | 45; 11 x 11 over 32, N = 64, 6272
// pixels 28.3 | 21.1 | 20.8), up to 512 tiles of 128 x 64 with two (9 x 9 over 48, N = 64, 25088 pixels: 26.9 against 32.0 with
// 64 x 64 and two); beyond those, and on K short of 32 stages, 128 x 128 behind more than 64 channels (K = 4096, N = 256, 25088
// pixels 44.6, as 64 x 64 69; K = 128, N = 256, 401408 pixels 77 | 101) and 256 x 64 for up to 64 from 65536 pixels on
// (K = 3872, 100352 pixels 60 against 92 as 64 x 64; K = 32, N = 48: 9.1 | 11.5, 50176 pixels level).
ConvGemmTile conv_walk_tile(int64_t M, int64_t N, int64_t stages) {
  const int64_t t64 = ceil_div(M, 64) * ceil_div(N, 64);
  if (stages >= 32 && t64 <= 512) return t64 <= 256 ? kConvGroups4 : kConvTall2;
  if (N > 64) return M >= 128 * 128 || stages >= 32 ? kConv128 : kConv64;
  return M >= 256 * 256 ? kConvRows256 : kConv64;
}

template <int MODE>
int launch_conv_gemm_walk(ConvGemmTile tile, const GemmArgs& a, const XConv& xs, hipStream_t s) {
  switch (tile) {
    case kConv64: return launch_conv_gemm_any_size<64, 64, 2, 2, MODE, false>(a, xs, s);
    case kConvGroups2: return launch_conv_gemm<64, 64, 2, 2, MODE, false, 2>(a, xs, s);
    case kConvGroups4: return launch_conv_gemm<64, 64, 2, 2, MODE, false, 4>(a, xs, s);
    case kConvTall2: return launch_conv_gemm<128, 64, 2, 2, MODE, false, 2>(a, xs, s);
    case kConvRows256: return launch_conv_gemm_any_size<256, 64, 4, 1, MODE, false>(a, xs, s);
    case kConv128: return launch_conv_gemm_any_size<128, 128, 2, 2, MODE, false>(a, xs, s);
    case kConv256: break;
  }
  return TMQ_ERR_UNSUPPORTED;
}

// The tile that tmq_conv2d_desc's tile_rows and tile_cols (wave groups) pin, if they do; false when there is none such.
// (The launch refuses what the table, or the walk, does not have.)
bool pinned_conv_tile(int32_t tile_rows, int32_t tile_cols, int64_t stages, ConvGemmTile* tile) {
  if (tile_rows <= 0 && tile_cols <= 0) return true;
  const int groups = tile_cols > 0 ? tile_cols : 1;
  if (stages % groups != 0) return false;
  if (tile_rows <= 0 && (groups == 1 || groups == 2 || groups == 4))
    *tile = groups == 1 ? kConv64 : groups == 2 ? kConvGroups2 : kConvGroups4;
  else if (tile_rows == 128 && (groups == 1 || groups == 2))
    *tile = groups == 1 ? kConv128 : kConvTall2;
  else if (tile_rows == 256 && groups == 1)
    *tile = kConv256;
  else
    return false;
  return true;
}

// Patch shape and LDS layout of the halo-tiled kernel for one problem.
struct TilePlan {
  int TH, TW, HH, HW, pitch, KS;
  int row_slots;  // 16-byte LDS slots per halo row, padding included
  int64_t rounds;  // of blocks, as many at once as fit the CUs' LDS
  int lds_x, lds_t, lds_tab, lds_total;
};

constexpr int kMaxDevices = 64;

int current_device() {
  int dev = 0;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices ? dev : -1;
}

// LDS bytes a block may use on the current device (cached per device; two
// threads that race on the first call store the same value).
int lds_limit() {
  static std::atomic<int> cache[kMaxDevices];
  const int dev = current_device();
  if (dev < 0) return 0;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// Chooses the patch that minimises a time estimate fitted to per-phase cycle
// stamps and a sweep of patch shapes at [32,56,56,64] x [64,3,3,64].  Per block:
//   fixed      3000 cycles of set-up, barriers and first-load latency
//   mfma       the busiest SIMD's row tiles x k-steps x 64 cycles
//   copy       weight bytes / 16 + 290 cycles per pass of the block over the halo
//              (a pass moves floor(512 / slots per halo row) whole halo rows, so
//              narrow halos waste fewer lanes: 28x14 patches take 5 passes where
//              7x56 patches of the same 392 pixels take 9)
//   epilogue   8.4 cycles per output pixel
// Blocks that fit a CU's LDS together overlap: the first costs the whole chain,
// each further one the larger of its SIMD work (half the fixed cost + mfma +
// epilogue) and its copies; blocks that do not fit run one after the other.  Returns false when
// the weight slice or the smallest halo do not fit.
bool plan_tiles(const ConvShape& s, bool forced, int forced_rows, int forced_cols, TilePlan* best) {
  // A block loads every pixel of its halo, so a kernel smaller than its stride
  // (1x1 stride 2: three of four loaded pixels unused) runs 1.6-3.7x faster as an
  // implicit GEMM, which gathers only what it multiplies.  Everything else that
  // fits is faster here, measured over ResNet-50's layer shapes at batch 32:
  // 3x3 stride 1 and 7x7 stride 2 by 1.8x, 3x3 stride 2 by 1.2-1.7x, 1x1 stride 1
  // by 1.05-1.8x.  With few output pixels and one round of blocks the wasted pixels cost
  // less than the implicit GEMM's long k loop on a handful of tiles (one image, 1x1 stride 2:
  // 256 -> 512 on 56 x 56 4.6 against 5.7 us, 1024 -> 2048 on 14 x 14 5.8 against 9.4 us; eight
  // images, 1024 -> 2048: 512 blocks, 17.6 against 9.7 us).
  const bool wasteful = !forced && s.KH * s.KW < s.sh * s.sw;
  if (wasteful && s.B * s.OH * s.OW > 1024) return false;
  const int64_t icb = s.ICg / 16;
  const int64_t chunks = s.KH * s.KW * icb;
  const int64_t KS = round_up(ceil_div(chunks, 2), 2);  // <= packed k-chunks / 2 (padded to 8)
  const int64_t w_bytes = 2048 * KS;
  const int64_t budget = static_cast<int64_t>(lds_limit()) - 3 * kCtBN * 4 - 256;
  if (w_bytes > 96 * 1024 || icb > 64) return false;
  const int64_t pitch = (icb | 1) * 16;
  const int64_t n_tiles = ceil_div(s.OCg, kCtBN);
  // patch widths: the whole row or a power of two, and the row cut into 2..8 equal parts
  int64_t widths[14];
  int nw = 0;
  const auto add_width = [&](int64_t w) {
    if (w < 1) return;
    for (int i = 0; i < nw; ++i)
      if (widths[i] == w) return;
    widths[nw++] = w;
  };
  if (forced_cols > 0) {
    add_width(s.OW < forced_cols ? s.OW : forced_cols);
  } else {
    for (int64_t cap : {128, 64, 32, 16, 8, 4}) add_width(s.OW < cap ? s.OW : cap);
    for (int64_t parts = 2; parts <= 8; ++parts) add_width(ceil_div(s.OW, parts));
  }
  double best_cost = -1.0;
  for (int wi = 0; wi < nw; ++wi) {
    const int64_t TW = widths[wi];
    const int64_t HWd = (TW - 1) * s.sw + (s.KW - 1) * s.dw + 1;
    // Slots per halo row.  A lane's pixel in the k loop is (r, c) of its row tile,
    // r = m / TW, c = m % TW for 32 consecutive m; consecutive pixels of one row lie
    // P = pitch / 16 (odd) slots apart, which spreads 16 lanes over the 16 slot
    // groups of the LDS, but a row tile crosses a patch row every TW lanes.  The
    // halo rows are padded so that the first pixel of the next row continues the
    // sequence: sh * row_slots = TW * sw * P (mod 16).  (Measured at
    // [32,56,56,64] x [64,3,3,64], 28 x 14 patches: bank-conflict cycles 443 k -> 210 k
    // per launch, LDS-active cycles 1.56 M -> 1.34 M; the launch time does not change,
    // the kernel is not bound by LDS bandwidth.)
    int64_t row_slots = HWd * (pitch / 16);
    for (int64_t pad = 0; pad < 16; ++pad)
      if ((s.sh * (row_slots + pad) - TW * s.sw * (pitch / 16)) % 16 == 0) {
        row_slots += pad;
        break;
      }
    if (row_slots > kCtThreads) continue;  // one halo row is copied in one pass of the block
    const int64_t rows_per_pass = kCtThreads / row_slots;
    for (int64_t TH = 1; TH <= s.OH && TH * TW <= kCtMaxPixels; ++TH) {
      if (forced_rows > 0 && TH != forced_rows) continue;
      const int64_t HH = (TH - 1) * s.sh + (s.KH - 1) * s.dh + 1;
      const int64_t x_bytes = HH * row_slots * 16;
      const int64_t total = w_bytes + x_bytes + kCtWaves * kCtTBytes + round_up(8 * (KS + 4), 16);
      if (total > budget) break;
      const int64_t blocks = s.B * ceil_div(s.OH, TH) * ceil_div(s.OW, TW) * n_tiles * s.groups;
      const int64_t MT = ceil_div(TH * TW, 32);
      const double mfma = static_cast<double>(ceil_div(MT, 4) * KS * 64);
      const double copy = static_cast<double>(w_bytes) / 16.0 + 290.0 * static_cast<double>(ceil_div(HH, rows_per_pass));
      const double epilogue = 8.4 * static_cast<double>(TH * TW);
      const int64_t per_cu = ceil_div(blocks, 256);
      int64_t together = kCuLds / (total + 3 * kCtBN * 4);
      together = together < 1 ? 1 : (together > per_cu ? per_cu : together);
      // half of the fixed cost is instructions (set-up, address tables), which a
      // co-resident block cannot hide
      const double simd = 1500.0 + mfma + epilogue;
      const double overlapped = simd > copy ? simd : copy;
      const double group = 3000.0 + mfma + copy + epilogue + static_cast<double>(together - 1) * overlapped;
      const double cost = static_cast<double>(ceil_div(per_cu, together)) * group;
      if (wasteful && blocks > 256) continue;
      if (best_cost < 0 || cost < best_cost) {
        best_cost = cost;
        best->TH = static_cast<int>(TH); best->TW = static_cast<int>(TW);
        best->HH = static_cast<int>(HH); best->HW = static_cast<int>(HWd);
        best->pitch = static_cast<int>(pitch); best->KS = static_cast<int>(KS);
        best->row_slots = static_cast<int>(row_slots);
        best->rounds = ceil_div(per_cu, together);
        best->lds_x = static_cast<int>(w_bytes);
        best->lds_t = static_cast<int>(w_bytes + x_bytes);
        best->lds_tab = best->lds_t + kCtWaves * kCtTBytes;
        best->lds_total = static_cast<int>(total);
      }
    }
  }
  return best_cost >= 0;
}

template <int MODE, int KIND, bool VEC>
int launch_conv_tiles_variant(const ConvShape& s, const TilePlan& p, const ConvTileArgs& a, hipStream_t stream) {
  // the kernel's LDS allowance is a per-device attribute: set once per device
  static std::atomic<uint64_t> done{0};
  const int dev = current_device();
  if (dev < 0) return TMQ_ERR_LAUNCH;
  if ((done.load(std::memory_order_acquire) >> dev & 1) == 0) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_tile_kernel<MODE, KIND, VEC>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds_limit() - 3 * kCtBN * 4) != hipSuccess)
      return TMQ_ERR_LAUNCH;
    done.fetch_or(uint64_t{1} << dev, std::memory_order_release);
  }
  const int64_t bx = s.B * a.tiles_h * a.tiles_w, by = static_cast<int64_t>(a.n_tiles) * s.groups;
  if (bx > 0x7fffffff || by > 65535) return TMQ_ERR_UNSUPPORTED;
  enqueue(conv_tile_kernel<MODE, KIND, VEC>,
          dim3(static_cast<unsigned>(bx), static_cast<unsigned>(by)), dim3(kCtThreads), p.lds_total, stream, a);
  return launch_status();
}

// Whether the packing conversion alone requantises this call's outputs (requant_plain_u8 of gemm_i8_core.h): zero
// point 0 and no bounds inside [0, 255] for unsigned bytes, the same 128 lower for signed ones.
template <int MODE>
bool plain_bytes(float zp_f, float lo_f, float hi_f) {
  const float shift = MODE == kOutS8 ? 128.f : 0.f;
  return requant_plain_u8(zp_f + shift, lo_f + shift, hi_f + shift);
}

// Which epilogue the launch needs (see conv_tile_kernel) is known on the host.
template <int MODE>
int launch_conv_tiles(const ConvShape& s, const TilePlan& p, const ConvTileArgs& a, hipStream_t stream) {
  const bool aligned16 = (reinterpret_cast<uintptr_t>(a.y) & 15) == 0;
  if constexpr (MODE == kOutAcc32) {
    const bool vec = (a.OC & 3) == 0 && (a.OCg & 3) == 0 && aligned16;
    return vec ? launch_conv_tiles_variant<MODE, 1, true>(s, p, a, stream)
               : launch_conv_tiles_variant<MODE, 1, false>(s, p, a, stream);
  } else {
    const bool vec = (a.OC & 15) == 0 && (a.OCg & 15) == 0 && aligned16;
    const int kind = a.post.silu ? 3
                     : a.post.accum != nullptr ? (plain_bytes<MODE>(a.zp_f, a.lo_f, a.hi_f) ? 5 : 0)
                     : plain_bytes<MODE>(a.zp_f, a.lo_f, a.hi_f) ? 4
                     : ((MODE == kOutU8 && a.lo_f <= 0.f && a.hi_f >= 255.f) ? 2 : 1);
    switch (kind * 2 + (vec ? 1 : 0)) {
      case 0: return launch_conv_tiles_variant<MODE, 0, false>(s, p, a, stream);
      case 1: return launch_conv_tiles_variant<MODE, 0, true>(s, p, a, stream);
      case 2: return launch_conv_tiles_variant<MODE, 1, false>(s, p, a, stream);
      case 3: return launch_conv_tiles_variant<MODE, 1, true>(s, p, a, stream);
      case 4: return launch_conv_tiles_variant<MODE, 2, false>(s, p, a, stream);
      case 5: return launch_conv_tiles_variant<MODE, 2, true>(s, p, a, stream);
      case 6: return launch_conv_tiles_variant<MODE, 3, false>(s, p, a, stream);
      case 7: return launch_conv_tiles_variant<MODE, 3, true>(s, p, a, stream);
      case 8: return launch_conv_tiles_variant<MODE, 4, false>(s, p, a, stream);
      case 9: return launch_conv_tiles_variant<MODE, 4, true>(s, p, a, stream);
      case 10: return launch_conv_tiles_variant<MODE, 5, false>(s, p, a, stream);
      default: return launch_conv_tiles_variant<MODE, 5, true>(s, p, a, stream);
    }
  }
}

// Tile shape and LDS use of the few-channel kernel (conv_runs.h) for one problem; false
// when the kernel does not take it: groups, dilation, kernel rows of more than 256 padded bytes.
struct RunPlan {
  int RL, RP, KS, TR, TW, mtw, rows_in, pitch, lds;
};
// The same for three channels as four-byte pixels (conv_image.h).  The cost of a schedule: rounds of tiles
// over the blocks the chip holds (three per CU) times a block's turns -- ten for each 16-pixel piece of its
// waves, two for each group of its threads, fifteen for the set-up of a round.
bool plan_image(const ConvShape& s, int forced_rows, RunPlan* p) {
  if (!s.pixels4 || s.B * s.H * s.W * 3 < 12) return false;
  constexpr int64_t kSlots = 3 * 256, kMaxGroups = int64_t{kCiUnits} * kCrThreads, kMaxLds = 48 * 1024;
  const int64_t by = ceil_div(s.OC, 16 * conv_runs_tiles(s.OC));
  int64_t best = -1;
  for (int64_t TW = s.OW < 256 ? s.OW : 256;; TW = round_up(TW / 2, 16)) {
    const int64_t mtw = ceil_div(TW, 16), G = ceil_div((TW - 1) * s.sw + s.runs_RP / 4, 4);
    for (int64_t TR = 1; TR <= s.OH && TR <= 16; ++TR) {
      const int64_t rows_in = (TR - 1) * s.sh + s.KH;
      if (rows_in * G > kMaxGroups || rows_in * G * 16 > kMaxLds) break;
      if (forced_rows > 0 && TR != forced_rows) continue;
      const int64_t tiles = s.B * ceil_div(s.OH, TR) * ceil_div(s.OW, TW);
      if (tiles > 0x7fffffff) continue;
      const int64_t cost = ceil_div(tiles * by, kSlots) *
                           (ceil_div(TR * mtw, kCrWaves) * 10 + ceil_div(rows_in * G, kCrThreads) * 2 + 15);
      if (best < 0 || cost < best) {
        best = cost;
        p->RL = static_cast<int>(s.runs_RL); p->RP = static_cast<int>(s.runs_RP); p->KS = static_cast<int>(s.runs_KS);
        p->TR = static_cast<int>(TR); p->TW = static_cast<int>(TW); p->mtw = static_cast<int>(mtw);
        p->rows_in = static_cast<int>(rows_in); p->pitch = static_cast<int>(G * 16);
        p->lds = static_cast<int>(rows_in * G * 16);
      }
    }
    if (TW <= 16) break;
  }
  return best >= 0;
}
bool plan_runs(const ConvShape& s, int forced_rows, RunPlan* p) {
  if (s.runs_KS == 0) return false;
  if (s.pixels4) return plan_image(s, forced_rows, p);
  const int64_t RL = s.runs_RL, RP = s.runs_RP, KS = s.runs_KS;
  // Tile = TR output rows x TW columns.  The staged image rows of a tile pass through
  // registers in units of 1 KB of a row, at most kCrUnits per wave; among the shapes that
  // fit, the one with the shortest schedule: rounds of tiles over the blocks the chip holds
  // (three per CU) times the turns its four waves need for the tile's 16-pixel pieces.
  constexpr int64_t kSlots = 3 * 256, kMaxUnits = int64_t{kCrUnits} * kCrWaves;
  int64_t best = -1;
  for (int64_t TW = s.OW < 128 ? s.OW : 128;; TW = round_up(TW / 2, 16)) {
    const int64_t mtw = ceil_div(TW, 16);
    const int64_t pitch = round_up((TW - 1) * s.sw * s.IC + RP + 20, 16);
    for (int64_t TR = 1; TR <= s.OH && TR <= 8; ++TR) {
      const int64_t rows_in = (TR - 1) * s.sh + s.KH;
      if (rows_in * ceil_div(pitch, 1024) > kMaxUnits) break;
      if (forced_rows > 0 && TR != forced_rows) continue;
      const int64_t tiles = s.B * ceil_div(s.OH, TR) * ceil_div(s.OW, TW);
      if (tiles > 0x7fffffff) continue;
      const int64_t cost = ceil_div(tiles, kSlots) * (ceil_div(TR * mtw, kCrWaves) * 10 + 5);
      if (best < 0 || cost < best) {
        best = cost;
        p->RL = static_cast<int>(RL); p->RP = static_cast<int>(RP); p->KS = static_cast<int>(KS);
        p->TR = static_cast<int>(TR); p->TW = static_cast<int>(TW); p->mtw = static_cast<int>(mtw);
        p->rows_in = static_cast<int>(rows_in); p->pitch = static_cast<int>(pitch);
        p->lds = static_cast<int>(rows_in * pitch);
      }
    }
    if (TW <= 16) break;
  }
  return best >= 0;
}

// Which layers' stores the L2s pass on at once (st16_through).  Off the 16-channel grid the lines are written in parts by
// different instructions, and each part goes to memory by itself (24 -> 40 channels on 32 x 56 x 56 5.9 -> 10.3 us).
int64_t out_bytes(const ConvShape& s) { return s.B * s.OH * s.OW * s.OC; }
bool lanes_on_grid(const ConvShape& s, const void* out) { return aligned(out, 16) && s.OC % (s.OC <= 32 ? 8 : 16) == 0; }
// From an image, of any size (us without | with them: 3 -> 64, 7 x 7, [32, 3, 224, 224] 19.4 | 15.9, one image 5.2 | 4.9;
// 3 -> 32, 3 x 3, 12.6 | 9.4 and 4.2 | 4.0), but for SiLU behind 7 x 7 and more than 32 channels short of 1 MiB, whose kernel
// waits for registers that it keeps in memory behind its stores (5.62 | 5.75).
bool image_through(const ConvShape& s, bool silu, const void* out) {
  return lanes_on_grid(s, out) && !(silu && s.KH * s.KW > 9 && s.OC > 32 && out_bytes(s) < int64_t{1} << 20);
}
// Pointwise rows: 64 -> 64 with a residual 6.4 MB 8.2 | 6.6, 64 -> 128 12.8 MB 13.1 | 10.0, 256 -> 128 12.5 | 10.7.  Where the
// lines leave the L2s during the kernel anyway, past 20 MB, those that several CUs write leave more than once (64 -> 384
// 38.5 MB 14.4 | 15.3); not so where a pixel's channel blocks are one CU's (64 -> 256 25.7 MB 15.2 | 14.4, 24 -> 512 19.7 |
// 18.9), nor where the kernel is no faster than the memory (SiLU: 64 -> 272 29.6 | 26.6, 256 -> 384 23.3 | 21.9; off the
// 64-channel grid up to 48 MiB, 208 -> 592 with a residual 85 MB 82 | 91).  Blocks that begin inside a line, past 12 MB (24 ->
// 112 11.2 MB 9.6 | 6.2, 24 -> 144 14.5 MB 9.9 | 11.2, 144 -> 864 18.3 MB 13.3 | 15.0).
// Nor for SiLU behind 65 to 128 channels short of 1 MiB: that kernel keeps five registers in memory and waits for them behind
// its stores (206 layers: 2.3 to 2.9 % behind below, level up to 2 MB, 2 to 7 % ahead from there; every other kernel is level
// below 0.25 MB and 2 to 11 % ahead from 2 MB on).
bool pointwise_through(const ConvShape& s, bool silu, const void* out) {
  const int64_t bytes = out_bytes(s);
  if (silu && s.runs_KS == 2 && bytes < int64_t{1} << 20) return false;
  const bool lines = s.OC % 64 == 0;
  return lanes_on_grid(s, out) &&
         (bytes <= int64_t{silu ? 48 : lines ? 20 : 12} << 20 || s.OC % 256 == 0 || (lines && (silu || s.runs_KS > 2)));
}
// Byte runs: the same from 2 MiB on, 2 to 4 % ahead; below level on average and up to 6 % behind (12 -> 16 on 8 x 96 x 97 1.2 MB
// 9.7 | 10.1, 24 -> 160 on 16 x 15 x 17 0.6 MB 7.9 | 8.4).
bool runs_through(const ConvShape& s, bool silu, const void* out) {
  return out_bytes(s) >= int64_t{2} << 20 && pointwise_through(s, silu, out);
}
// Halo tiles: a block has 64 channels of its pixels.  64 -> 64 on 32 x 56 x 56 11.6 | 10.2, on 16 x 56 x 56 7.2 | 6.7, one
// image 5.2 | 5.1; where other blocks write the rest of a line, up to 8 MB (96 channels 4.8 MB 11.3 | 9.7, 9.6 MB 16.8 | 17.4).
bool tiles_through(const ConvShape& s, const void* out) {
  return aligned(out, 16) && s.OC % 16 == 0 && (s.OC <= 64 || s.OC % 64 == 0 || out_bytes(s) <= int64_t{8} << 20);
}
// Depthwise, four bytes a lane: 96 channels on 4 x 56 x 56 1.2 MB 4.9 | 5.4, 60 on 32 x 56 x 56 6 MB 10.0 | 8.4, 144 on
// 16 x 56 x 56 7.2 MB 11.1 | 9.6, 192 on 32 x 56 x 56 19.3 MB 15.3 | 15.8.  Not where the arithmetic covers the stores: 7 x 7 is
// level (relu) and 1 % behind (SiLU), 5 x 5 with SiLU level on average and up to 6 % behind (448 channels on 2 x 80 x 75 14.6 |
// 15.4); 5 x 5 without is 2 to 4 % ahead.
bool depthwise_through(const ConvShape& s, bool silu, const void* out) {
  const int64_t bytes = out_bytes(s);
  return aligned(out, 4) && s.OC % 4 == 0 && bytes >= int64_t{9} << 19 && bytes <= int64_t{16} << 20 && s.KH == s.KW &&
         (s.KH == 3 || (s.KH == 5 && !silu));
}

template <int MODE>
int launch_conv_runs(const tmq_conv2d_desc* d, const ConvShape& s, const RunPlan& p, const PostOps& po, float zp_f,
                     float lo_f, float hi_f, void* out, hipStream_t stream) {
  ConvRunArgs a{};
  a.x = static_cast<const uint8_t*>(d->x);
  a.w_runs = static_cast<const uint8_t*>(d->w_packed) + s.runs_off;
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.bias = d->bias;
  a.y = out;
  a.B = static_cast<int>(s.B);
  a.H = static_cast<int>(s.H); a.W = static_cast<int>(s.W); a.IC = static_cast<int>(s.IC);
  a.OH = static_cast<int>(s.OH); a.OW = static_cast<int>(s.OW); a.OC = static_cast<int>(s.OC);
  a.KH = static_cast<int>(s.KH); a.KW = static_cast<int>(s.KW);
  a.sh = static_cast<int>(s.sh); a.sw = static_cast<int>(s.sw);
  a.ph = static_cast<int>(s.ph); a.pw = static_cast<int>(s.pw);
  a.RL = p.RL; a.RP = p.RP; a.KS = p.KS;
  a.TR = p.TR; a.TW = p.TW; a.mtw = p.mtw;
  a.rows_in = p.rows_in; a.pitch = p.pitch;
  a.tiles_h = static_cast<int>(ceil_div(s.OH, p.TR));
  a.tiles_w = static_cast<int>(ceil_div(s.OW, p.TW));
  a.tiles = static_cast<int32_t>(s.B * a.tiles_h * a.tiles_w);
  if constexpr (MODE == kOutAcc32)
    a.vec = aligned(out, 16) && s.OC % 4 == 0 ? 1 : 0;
  else
    a.through = (s.pixels4 ? image_through(s, po.silu, out) : runs_through(s, po.silu, out)) ? 1 : 0;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.x_xor = d->x_signed ? 0u : 0x80808080u;
  a.pad_word = 0x01010101u * static_cast<uint32_t>(static_cast<uint8_t>(d->x_zero_point));
  a.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.out_scale = d->out_scale;
  a.zp_f = zp_f; a.lo_f = lo_f; a.hi_f = hi_f;
  a.post = po;
  const int nt = conv_runs_tiles(s.OC);
  const int64_t by = ceil_div(s.OC, 16 * nt);
  if (by > 65535) return TMQ_ERR_UNSUPPORTED;
  // three blocks per CU (their registers), each with its weights in registers for every tile it walks
  const int64_t slots = s.pixels4 ? std::max<int64_t>(768 / by, 1) : 768;  // (plan_runs, plan_image: kSlots)
  const int64_t bx = a.tiles < slots ? a.tiles : slots;
  const dim3 grid(static_cast<unsigned>(bx), static_cast<unsigned>(by)), block(kCrThreads);
  const auto launch = [&](auto post_tag, auto nt_tag, auto plain_tag) {
    constexpr int kP = decltype(post_tag)::value, kNT = decltype(nt_tag)::value;
    constexpr bool kPlain = decltype(plain_tag)::value;
    const auto image = [&](auto ks_tag) {
      constexpr int kKS = decltype(ks_tag)::value;
      if (s.sw % 2 == 0)
        enqueue(conv_image_kernel<MODE, kP, kNT, kKS, true, kPlain>, grid, block, p.lds, stream, a);
      else
        enqueue(conv_image_kernel<MODE, kP, kNT, kKS, false, kPlain>, grid, block, p.lds, stream, a);
    };
    if (s.pixels4 && s.runs_KS == 1)
      image(std::integral_constant<int, 1>{});
    else if (s.pixels4)
      image(std::integral_constant<int, kCrMaxKS>{});
    else
      enqueue(conv_runs_kernel<MODE, decltype(post_tag)::value, decltype(nt_tag)::value, decltype(plain_tag)::value>, grid, block, p.lds, stream, a);
  };
  const auto launch_tiles = [&](auto nt_tag) {
    if constexpr (MODE != kOutAcc32) {
      const bool plain = plain_bytes<MODE>(zp_f, lo_f, hi_f);
      if (po.silu) return launch(std::integral_constant<int, 2>{}, nt_tag, std::false_type{});
      if (po.any() && plain) return launch(std::integral_constant<int, 1>{}, nt_tag, std::true_type{});
      if (po.any()) return launch(std::integral_constant<int, 1>{}, nt_tag, std::false_type{});
      if (plain) return launch(std::integral_constant<int, 0>{}, nt_tag, std::true_type{});
    }
    launch(std::integral_constant<int, 0>{}, nt_tag, std::false_type{});
  };
  if (nt == 2)
    launch_tiles(std::integral_constant<int, 2>{});
  else
    launch_tiles(std::integral_constant<int, 4>{});
  return launch_status();
}

// Pointwise layers over at most 256 input channels with their pixels straight from memory
// (conv_runs_pointwise_kernel); false when the layer is not one of them.
bool pointwise_rows_ok(const tmq_conv2d_geom& g, const ConvShape& s) {
  return g.groups == 1 && s.KH == 1 && s.KW == 1 && s.sh == 1 && s.sw == 1 && s.ph == 0 && s.pw == 0 && s.runs_KS > 0 &&
         s.B * s.H * s.W <= 0x7fffff00 && s.B * s.H * s.W * s.IC >= 16 && s.OC <= 65536;
}

// Where it is ahead of everything else that runs the layer (us, it | the best other): with a residual or SiLU (batch 32,
// 256 -> 512 on 28 x 28 15.1 | 18.6; 128 -> 768 on 53 x 109 at batch 6 17.7 | 28.8; one image, 96 -> 576 on 14 x 14 4.4 | 5.3),
// up to 128 input channels (batch 32: 128 -> 512 on 28 x 28 10.6 | 10.8; one image: 64 -> 256 on 56 x 56 4.2 | 4.5) and up to
// 32 output channels (144 -> 24 on one image of 57 x 43 4.2 | 4.7).  Of more of both, against the linear kernels, by the
// pieces of 16 pixels times the blocks of 64 channels: up to 1024, one for each SIMD (208 -> 1024 on 560 pixels 3.65 | 3.9,
// 192 -> 192 on 4899 3.5 | 3.9), and again from where the linear kernels are past what they do at once: 2048, or 3072 where
// more than four channel blocks read the same pixels (192 -> 128 on 50176 6.9 | 7.4, 208 -> 1024 on 9792 8.7 | 11.4; in between
// 240 -> 64 on 25088 4.65 | 4.4, 192 -> 960 on 2812 5.4 | 5.1); over 256 channels, whole 128-byte lines to the linear kernels,
// 8192, or 4096 for one block (256 -> 512 on 4761 6.2 | 5.1, on 21312 10.8 | 11.6; 256 -> 64 on 50176 6.7 | 6.4, on 100352 8.4 |
// 9.3).  On 570 random layers the choice is 0.1 % behind the better of the two on average and 7 % at most.
bool pointwise_rows_first(const ConvShape& s, bool post) {
  if (post || s.runs_KS <= 2 || s.OC <= 32) return true;
  const int64_t blocks = ceil_div(s.OC, 64), units = ceil_div(s.B * s.H * s.W, 16) * blocks;
  return units <= 1024 || units > (s.IC == 256 ? (blocks == 1 ? 4096 : 8192) : blocks <= 4 ? 2048 : 3072);
}

// The 16-pixel pieces whose reads and stores the kernel makes without a check: all 16 pixels exist, and the last pixel's
// 16-byte reads (to RP >= IC bytes behind its first) end inside the tensor.  None where a lane's residual bytes are more
// than a pixel has.
int64_t pointwise_whole_pieces(int64_t pixels, int64_t IC, int64_t RP, bool short_residual) {
  const int64_t last = pixels * IC - RP - 15 * IC;  // first byte of the last piece that may be read so
  if (short_residual || last < 0) return 0;
  return std::min(pixels / 16, last / (16 * IC) + 1);
}

template <int MODE>
int launch_conv_pointwise_rows(const tmq_conv2d_desc* d, const ConvShape& s, const PostOps& po, float zp_f, float lo_f,
                               float hi_f, void* out, hipStream_t stream) {
  ConvRunArgs a{};
  a.x = static_cast<const uint8_t*>(d->x);
  a.w_runs = static_cast<const uint8_t*>(d->w_packed) + s.runs_off;
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.bias = d->bias;
  a.y = out;
  a.B = static_cast<int>(s.B);
  a.H = static_cast<int>(s.H); a.W = static_cast<int>(s.W); a.IC = static_cast<int>(s.IC);
  a.OH = static_cast<int>(s.OH); a.OW = static_cast<int>(s.OW); a.OC = static_cast<int>(s.OC);
  a.KH = a.KW = 1;
  a.sh = a.sw = 1;
  a.RL = static_cast<int>(s.runs_RL); a.RP = static_cast<int>(s.runs_RP); a.KS = static_cast<int>(s.runs_KS);
  const int64_t pieces = ceil_div(s.B * s.H * s.W, 16);
  a.tiles = static_cast<int32_t>(pieces);
  if constexpr (MODE == kOutAcc32) a.vec = aligned(out, 16) && s.OC % 4 == 0 ? 1 : 0;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.x_xor = d->x_signed ? 0u : 0x80808080u;
  a.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.out_scale = d->out_scale;
  a.zp_f = zp_f; a.lo_f = lo_f; a.hi_f = hi_f;
  a.post = po;
  const int nt = conv_runs_tiles(s.OC);
  a.whole = static_cast<int32_t>(pointwise_whole_pieces(s.B * s.H * s.W, s.IC, s.runs_RP, po.accum != nullptr && s.OC < 4 * nt));
  // one wave per channel block and run of pieces, as many as the chip holds at once (their registers), but at least
  // one per channel block
  const int64_t nblk = ceil_div(s.OC, 16 * nt), cap = 256 * (s.runs_KS > 2 ? 2 : 3) * kCrWaves;
  int64_t groups = cap / nblk < 1 ? 1 : cap / nblk;
  if (groups > pieces) groups = pieces;
  // groups dealt to the XCDs where some have a piece more than the rest, as many to each if that costs no further piece
  const bool by_xcd = nblk >= kCrXcdBlocks;
  const int64_t even = groups - groups % 8;
  const bool deal = by_xcd && groups >= 8 && pieces % groups != 0 && ceil_div(pieces, even) == ceil_div(pieces, groups);
  if (deal) groups = even;
  const int64_t blocks = deal ? 8 * ceil_div(ceil_div(groups, 8) * nblk, kCrWaves) : ceil_div(groups * nblk, kCrWaves);
  a.nblk = static_cast<int>(nblk);
  a.groups = static_cast<int>(groups);
  // (exact while waves x nblk < 2**32: at most 3072 waves, or nblk <= 2048 of them)
  a.nblk_magic = static_cast<uint32_t>(((int64_t{1} << 32) + nblk - 1) / nblk);
  a.xcd_mask = by_xcd ? 7 : 0;
  a.xcd_shift = by_xcd ? 3 : 0;
  a.xcd_blocks = by_xcd && !deal ? static_cast<uint32_t>(blocks / 8) : 0;
  a.xcd_longer = by_xcd && !deal ? static_cast<uint32_t>(blocks % 8) : 0;
  a.deal_shift = deal ? 3 : 0;
  a.deal_mask = deal ? 7 : 0;
  const dim3 grid(static_cast<unsigned>(blocks)), block(kCrThreads);
  const auto launch_as = [&](auto post_tag, auto nt_tag, auto plain_tag, auto through_tag) {
    constexpr int kP = decltype(post_tag)::value, kNT = decltype(nt_tag)::value;
    constexpr bool kPlain = decltype(plain_tag)::value, kThrough = decltype(through_tag)::value;
    if (s.runs_KS == 1)
      enqueue(conv_runs_pointwise_kernel<MODE, kP, kNT, 1, kPlain, kThrough>, grid, block, 0, stream, a);
    else if (s.runs_KS == 2)
      enqueue(conv_runs_pointwise_kernel<MODE, kP, kNT, 2, kPlain, kThrough>, grid, block, 0, stream, a);
    else
      enqueue(conv_runs_pointwise_kernel<MODE, kP, kNT, 4, kPlain, kThrough>, grid, block, 0, stream, a);
  };
  const auto launch = [&](auto post_tag, auto nt_tag, auto plain_tag) {
    if constexpr (MODE != kOutAcc32) {
      if (pointwise_through(s, po.silu, out)) return launch_as(post_tag, nt_tag, plain_tag, std::true_type{});
    }
    launch_as(post_tag, nt_tag, plain_tag, std::false_type{});
  };
  const auto launch_tiles = [&](auto nt_tag) {
    if constexpr (MODE != kOutAcc32) {
      const bool plain = plain_bytes<MODE>(zp_f, lo_f, hi_f);
      if (po.silu) return launch(std::integral_constant<int, 2>{}, nt_tag, std::false_type{});
      if (po.any() && plain) return launch(std::integral_constant<int, 1>{}, nt_tag, std::true_type{});
      if (po.any()) return launch(std::integral_constant<int, 1>{}, nt_tag, std::false_type{});
      if (plain) return launch(std::integral_constant<int, 0>{}, nt_tag, std::true_type{});
    }
    launch(std::integral_constant<int, 0>{}, nt_tag, std::false_type{});
  };
  if (nt == 2)
    launch_tiles(std::integral_constant<int, 2>{});
  else
    launch_tiles(std::integral_constant<int, 4>{});
  return launch_status();
}

// Depthwise layers on the vector ALU (conv_depthwise.h).
template <int MODE>
int launch_conv_depthwise(const tmq_conv2d_desc* d, const ConvShape& s, const PostOps& po, float zp_f, float lo_f,
                          float hi_f, void* out, hipStream_t stream) {
  DepthwiseArgs a{};
  a.x = static_cast<const uint8_t*>(d->x);
  a.w_taps = static_cast<const uint8_t*>(d->w_packed) + s.runs_off;
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.bias = d->bias;
  a.y = out;
  a.B = static_cast<int>(s.B);
  a.H = static_cast<int>(s.H); a.W = static_cast<int>(s.W); a.C = static_cast<int>(s.IC);
  a.OH = static_cast<int>(s.OH); a.OW = static_cast<int>(s.OW);
  a.KH = static_cast<int>(s.KH); a.KW = static_cast<int>(s.KW);
  a.sh = static_cast<int>(s.sh); a.sw = static_cast<int>(s.sw);
  a.ph = static_cast<int>(s.ph); a.pw = static_cast<int>(s.pw);
  a.dh = static_cast<int>(s.dh); a.dw = static_cast<int>(s.dw);
  // Output rows per lane: long strips amortise the lane's weights and constants, short ones put
  // more waves in flight; the longest with a wave per SIMD (half a wave under a 7 x 7 kernel, whose
  // window of 49 taps is the larger part of a short strip's work).
  // Under 5 x 5 and 7 x 7 windows, whose first rows are the larger part of a short strip, up to 14 rows, and the
  // image in equal strips (7 x 7 over 96 channels on 56 x 56: 21.1 -> 18.9 us; 5 x 5 over 240 channels on 28 x 28:
  // 12.6 -> 10.8 us; 3 x 3 gains nothing beyond 8).
  const bool pinned_strip = d->kernel == 7 && d->tile_rows > 0;
  int64_t strip = pinned_strip ? d->tile_rows : kDwStripMax;
  // (images of 9 to 14 rows in two strips: 5 x 5 over 672 channels on 14 x 14 9.9 against 10.8 us in one)
  if (!pinned_strip && s.KH >= 5 && s.OH > 8) strip = ceil_div(s.OH, s.OH <= 14 ? 2 : ceil_div(s.OH, 14));
  // Two columns a lane for 3 x 3 at stride 1 where strips of eight rows are four waves a SIMD and more of one column (us, one | two: 624
  // channels on 15 x 42 x 26 12.3 | 10.7, 768 on 15 x 55 x 27 17.6 | 15.1, 864 on 28 x 100 x 44 85 | 72; with the layers around it,
  // 768 on 14 x 26 x 59 33.4 | 29.8, 816 on 4 x 106 x 74 56.7 | 53.2, 288 on 23 x 69 x 53 46.1 | 44.4; below, what is left over of the
  // last wave decides, 288 on 25 x 7 x 110 23.1 | 23.8).  From 256 channels on: fewer leave a line in two parts, which what follows pays
  // for (234 on 15 x 33 x 97 30.5 | 31.4, 120 on 27 x 38 x 69 32.1 | 33.0); and no odd width that wastes more than a sixteenth (768 on
  // 18 x 55 x 13 30.1 | 30.4).
  const bool pairs = !pinned_strip && s.KH == 3 && s.KW == 3 && s.sh == 1 && s.sw == 1 && s.dh == 1 && s.dw == 1 && s.IC >= 256 &&
                     (s.OW % 2 == 0 || s.OW > 16) &&
                     s.B * ceil_div(s.OH, kDwStripMax) * s.OW * ceil_div(s.IC, 4) >= int64_t{1} << 18;
  const int64_t across = pairs ? ceil_div(s.OW, 2) : s.OW;
  const int64_t lanes_wanted = int64_t{1} << (s.KH == 7 && s.KW == 7 ? 15 : 16);
  if (!pinned_strip)
    while (strip > 1 && s.B * ceil_div(s.OH, strip) * across * ceil_div(s.IC, 4) < lanes_wanted) strip = ceil_div(strip, 2);
  if (strip > s.OH) strip = s.OH;
  a.strip = static_cast<int>(strip);
  const int64_t per_image = ceil_div(s.OH, strip) * across * ceil_div(s.IC, 4);
  const int64_t blocks_per_image = ceil_div(per_image, kDwThreads);
  a.per_image = static_cast<uint32_t>(per_image);
  a.blocks_per_image = static_cast<uint32_t>(blocks_per_image);
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.x_xor = d->x_signed ? 0u : 0x80808080u;
  a.pad_word = 0x01010101u * static_cast<uint32_t>(static_cast<uint8_t>(d->x_zero_point));
  a.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.out_scale = d->out_scale;
  a.zp_f = zp_f; a.lo_f = lo_f; a.hi_f = hi_f;
  a.post = po;
  const int64_t blocks = s.B * blocks_per_image;
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>(blocks)), block(kDwThreads);
  const auto launch_as = [&](auto post_tag, auto through_tag) {
    constexpr bool kP = decltype(post_tag)::value, kThrough = decltype(through_tag)::value;
    if (pairs)
      enqueue(conv_depthwise_kernel<MODE, kP, 3, kThrough, 2>, grid, block, 0, stream, a);
    else if (s.KH == 3 && s.KW == 3)
      enqueue(conv_depthwise_kernel<MODE, kP, 3, kThrough>, grid, block, 0, stream, a);
    else if (s.KH == 5 && s.KW == 5)
      enqueue(conv_depthwise_kernel<MODE, kP, 5, kThrough>, grid, block, 0, stream, a);
    else if (s.KH == 7 && s.KW == 7)
      enqueue(conv_depthwise_kernel<MODE, kP, 7, false>, grid, block, 0, stream, a);
    else
      enqueue(conv_depthwise_kernel<MODE, kP, 0, false>, grid, block, 0, stream, a);
  };
  const auto launch = [&](auto post_tag) {
    if constexpr (MODE != kOutAcc32) {
      if (depthwise_through(s, po.silu, out)) return launch_as(post_tag, std::true_type{});
    }
    launch_as(post_tag, std::false_type{});
  };
  if constexpr (MODE != kOutAcc32) {
    if (po.any()) {
      launch(std::true_type{});
      return launch_status();
    }
  }
  launch(std::false_type{});
  return launch_status();
}

// quantized::linear over `rows` rows of K bytes at `x` (the pixels of a pointwise layer, or patch
// rows) with the layer's packed weight, which for one group over whole 16-channel blocks is the
// linear layout: [OC, K] in 16-channel blocks, k = (kh, kw, ic).
int run_as_linear(const tmq_conv2d_desc* d, int64_t rows, int64_t OC, int64_t K, const void* x, bool relu, void* out,
                  hipStream_t stream) {
  tmq_linear_desc l{};
  l.M = rows; l.N = OC; l.K = K;
  l.x = x; l.ldx = K;
  l.x_signed = d->x_signed; l.x_zero_point = d->x_zero_point; l.x_scale = d->x_scale;
  l.w_packed = d->w_packed; l.w_colsum = d->w_colsum; l.w_scales = d->w_scales;
  l.w_per_channel = d->w_per_channel;
  l.relu = relu ? 1 : 0;
  l.bias = d->bias;
  l.out_scale = d->out_scale; l.out_zero_point = d->out_zero_point; l.out_signed = d->out_signed;
  l.y = out; l.ldy = OC;
  return tmq_linear(&l, reinterpret_cast<tmq_stream_t>(stream));
}

// Operands of the implicit GEMM (of a layer's first group).
void conv_gemm_operands(const tmq_conv2d_desc* d, const ConvShape& s, const PostOps& po, float zp_f, float lo_f, float hi_f,
                        void* out, GemmArgs* args, XConvTable* source) {
  XConvTable& xs = *source;
  xs.x = static_cast<const uint8_t*>(d->x);
  xs.H = static_cast<int>(s.H); xs.W = static_cast<int>(s.W); xs.IC = static_cast<int>(s.IC);
  xs.OH = static_cast<int>(s.OH); xs.OW = static_cast<int>(s.OW);
  xs.KW = static_cast<int>(s.KW); xs.icb = static_cast<int>(s.ICgp / 16);
  xs.stride_h = static_cast<int>(s.sh); xs.stride_w = static_cast<int>(s.sw);
  xs.pad_h = static_cast<int>(s.ph); xs.pad_w = static_cast<int>(s.pw);
  xs.dil_h = static_cast<int>(s.dh); xs.dil_w = static_cast<int>(s.dw);
  xs.pad_word = 0x01010101u * static_cast<uint32_t>(static_cast<uint8_t>(d->x_zero_point));
  xs.KH = static_cast<int>(s.KH);
  xs.chunks = static_cast<int>(s.Kp / 16);
  xs.step_w = static_cast<int>(s.dw * s.IC - 16 * (s.ICgp / 16));
  xs.step_h = static_cast<int>(s.dh * s.W * s.IC - s.KW * s.dw * s.IC);

  GemmArgs& a = *args;
  a.M = s.B * s.OH * s.OW;
  a.N = s.OCg;
  a.K = s.Kp;
  a.w_packed = static_cast<const uint8_t*>(d->w_packed);
  a.w_kchunks = s.KC;
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.bias = d->bias;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.x_xor = d->x_signed ? 0u : 0x80808080u;
  a.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.out_scale = d->out_scale;
  a.zp_f = zp_f; a.lo_f = lo_f; a.hi_f = hi_f;
  a.y = out;
  a.ldy = s.OC;
  a.post = po;
}

template <int MODE>
int launch_conv_waves(const GemmArgs& a, const XConvTable& xs, int tile, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(ceil_div(a.N, tile)), static_cast<unsigned>(ceil_div(a.M, 32)));
  if (tile == 32) enqueue(gemm_i8_wloop_kernel<MODE, 1, XConvTable>, grid, dim3(kWloopWaves * kWave), 0, s, a, xs);
  else enqueue(gemm_i8_wloop_kernel<MODE, 2, XConvTable>, grid, dim3(kWloopWaves * kWave), 0, s, a, xs);
  return launch_status();
}
// Layers of one group whose pixels and channels make one round of tiles of 32 rows: their eight waves walk K in pieces, the windows'
// chunks gathered straight into registers (gemm_i8_wloop.h).  Everything else that takes such a layer has a chain as long as K on a
// few blocks, or a copy in front: us, the best before | these, 3 x 3: 512 -> 398 on 8 x 9 x 10 15.2 | 9.6, 256 -> 256 on one 28 x 28
// 9.4 | 6.0, 512 -> 512 on one 14 x 14 (patch rows) 14.6 | 7.0, 192 -> 192 on 2 x 20 x 67 8.7 | 7.0, 112 -> 48 with SiLU on 8 x 10 x 19 (halo
// tiles) 6.9 | 4.8; 1 x 1 with SiLU, 624 -> 304 on 2 x 24 x 23 6.5 | 5.5; 960 -> 187 with SiLU on 3 x 7 x 34 22.7 | 10.4.  Of 240 drawn
// layers (K = 144 ... 23040) 32 channels a tile take 0.40 to 0.98 of the time where they fit a round, but for K short of 576 without
// a residual or SiLU (0.96 to 1.13, halo tiles and patches in registers); 64 channels, where only those fit, 0.56 to 0.99 from K = 720
// (400 with a residual or SiLU) on, below 0.86 to 1.2.  A second round is behind: 1.0 to 1.9.
// Returns the channels per tile, 0: not such a layer.
int conv_waves_tile(const ConvShape& s, const tmq_conv2d_geom& g, bool post) {
  if (g.groups != 1 || s.groups != 1 || s.ICg % 16 != 0 || !conv_table_takes(s)) return 0;
  const int64_t rows = ceil_div(s.B * s.OH * s.OW, 32);
  if (rows * ceil_div(s.OC, 32) <= 256) return post || s.Kp >= 576 ? 32 : 0;
  return rows * ceil_div(s.OC, 64) <= 256 && s.Kp >= (post ? 400 : 720) ? 64 : 0;
}

template <int MODE>
int run_conv(const tmq_conv2d_desc* d, const tmq_conv2d_post* post, void* out, hipStream_t stream) {
  ConvShape s;
  int rc = make_shape(&d->geom, &s);
  if (rc != TMQ_OK) return rc;
  const int64_t rows = s.B * s.OH * s.OW;
  if (rows == 0) return TMQ_OK;
  if (d->x == nullptr || d->w_packed == nullptr || d->w_colsum == nullptr || out == nullptr)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(d->w_packed, 16)) return TMQ_ERR_ALIGNMENT;
  const int qmin = d->out_signed ? -128 : 0, qmax = d->out_signed ? 127 : 255;
  const int xmin = d->x_signed ? -128 : 0, xmax = d->x_signed ? 127 : 255;
  if (d->x_zero_point < xmin || d->x_zero_point > xmax) return TMQ_ERR_INVALID_ARGUMENT;
  if (MODE != kOutAcc32) {
    if (d->w_scales == nullptr || !(d->x_scale > 0.f) || !(d->out_scale > 0.f))
      return TMQ_ERR_INVALID_ARGUMENT;
    if (d->out_zero_point < qmin || d->out_zero_point > qmax) return TMQ_ERR_INVALID_ARGUMENT;
  }
  PostOps po{};
  bool relu = d->relu != 0;
  if (post != nullptr) {
    if (MODE == kOutAcc32) return TMQ_ERR_INVALID_ARGUMENT;
    if (post->activation < 0 || post->activation > 2) return TMQ_ERR_INVALID_ARGUMENT;
    if (post->activation == 2 && relu) return TMQ_ERR_INVALID_ARGUMENT;
    relu = relu || post->activation == 1;
    po.silu = post->activation == 2;
    po.out_scale = d->out_scale;
    {
      const double exact = -static_cast<double>(d->out_scale) * 1.4426950408889634074;  // -s log2(e)
      po.silu_c = static_cast<float>(exact);
      po.silu_c_tail = static_cast<float>(exact - static_cast<double>(po.silu_c));
    }
    if (post->accum != nullptr) {
      const int amin = post->accum_signed ? -128 : 0, amax = post->accum_signed ? 127 : 255;
      if (!(post->accum_scale > 0.f) || post->accum_zero_point < amin || post->accum_zero_point > amax)
        return TMQ_ERR_INVALID_ARGUMENT;
      po.accum = static_cast<const uint8_t*>(post->accum);
      po.accum_signed = post->accum_signed;
      po.accum_zp = post->accum_zero_point;
      po.amult = post->accum_scale / d->out_scale;
    }
  }
  const float zp_f = static_cast<float>(d->out_zero_point);
  const float lo_f = static_cast<float>(relu ? d->out_zero_point : qmin);
  const float hi_f = static_cast<float>(qmax);

  const int forced = d->kernel > 0 ? d->kernel : -1;
  // A pointwise layer (1 x 1, stride 1, no padding, one group) is a linear layer over the
  // pixels: rows = pixels, K = input channels, and the packed weight is the linear one
  // (same 16-channel blocks, same k padding), and the linear kernels take it unless pointwise_rows_first says otherwise:
  // over more than 256 channels the best other kernel took 1.11 to 1.5 times as long on most of 180 random layers (288 -> 64
  // on 23326 pixels 5.0 | 4.5 us, 512 -> 64 on 20880 5.7 | 4.9, 640 -> 32 on 46176 8.5 | 6.7, 768 -> 80 on 8460 6.0 | 5.1, 1024
  // -> 112 on 8844 7.7 | 6.0, 1024 -> 256 on 14 x 14 at batch 32 12.8 | 7.8); where it was ahead (272 -> 48 on 102144 8.7 | 9.2),
  // by 5 % at most.
  if constexpr (MODE != kOutAcc32) {
    const bool pointwise = s.KH == 1 && s.KW == 1 && s.sh == 1 && s.sw == 1 && s.ph == 0 && s.pw == 0 &&
                           d->geom.groups == 1 && s.IC % 16 == 0 && aligned(d->x, 16) && !po.any();
    if (forced == 5 && !pointwise) return TMQ_ERR_UNSUPPORTED;
    if (forced == 5 || (forced < 0 && pointwise && !(pointwise_rows_ok(d->geom, s) && pointwise_rows_first(s, false)))) {
      return run_as_linear(d, rows, s.OC, s.IC, d->x, relu, out, stream);
    }
  }
  if constexpr (MODE != kOutAcc32) {
    const int tile = forced < 0 && aligned(d->x, 16) ? conv_waves_tile(s, d->geom, po.any()) : 0;
    if (tile != 0 && !(pointwise_rows_ok(d->geom, s) && pointwise_rows_first(s, po.any()))) {
      GemmArgs a{};
      XConvTable xs{};
      conv_gemm_operands(d, s, po, zp_f, lo_f, hi_f, out, &a, &xs);
      return launch_conv_waves<MODE>(a, xs, tile, stream);
    }
  }
  // Few output pixels against a long K and a weight slice the halo tiles cannot hold: with a
  // workspace the patch rows are written out and the product runs on the linear kernels
  // (3 x 3 at 196 pixels, patch rows | implicit GEMM with its wave groups: 256 -> 256 channels 8.9 | 9.5 us, 384 -> 384
  // 10.3 | 11.8, 448 -> 448 10.4 | 13.3, 512 -> 512 16.2 | 14.2; at 480: 384 -> 384 11.8 | 11.8, 512 -> 512 17.5 | 14.3;
  // 1024 -> 1024 at 196 26.7 | 22.3, at 49 19.8 | 21.9; 512 -> 512 at 49 14.1 | 14.0; layers that walk: 8 x 8, 256 -> 256 at
  // 196 37.3 | 42.1, 11 x 11, 96 -> 96 at 196 29.4 | 31.8, at 784 34.5 | 32.4; 11 x 11, 32 -> 64 at 784 11.7 | 20.0, at 3136
  // 21.3 | 20.6, 8 x 8, 64 -> 256 at 784 15.0 | 16.0, at 1568 18.3 | 16.3).
  if constexpr (MODE != kOutAcc32) {
    if (forced == 6 || forced < 0) {
      const int64_t need = po.any() || !aligned(d->x, 16) ? 0 : patch_rows_bytes(d->geom, s, forced == 6);
      TilePlan tp;
      const bool use = need > 0 && d->workspace != nullptr && d->workspace_bytes >= need && aligned(d->workspace, 16) &&
                       (forced == 6 || !plan_tiles(s, false, 0, 0, &tp));
      if (forced == 6 && !use) return TMQ_ERR_UNSUPPORTED;
      if (use) {
        const int64_t chunks = need / 16;
        enqueue(conv_patch_rows_kernel, dim3(static_cast<unsigned>(ceil_div(chunks, 256))), dim3(256), 0, stream,
                static_cast<const uint8_t*>(d->x), s, chunks,
                0x01010101u * static_cast<uint32_t>(static_cast<uint8_t>(d->x_zero_point)), static_cast<uint8_t*>(d->workspace));
        if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
        return run_as_linear(d, rows, s.OC, s.Kp, d->workspace, relu, out, stream);
      }
    }
  }
  // Channel counts off the 16-channel grid under kernel rows too long for the byte runs: the MFMA kernels on a
  // padded copy of the input in the caller's scratch memory (3 x 3, 40 -> 40 channels on 56 x 56 at batch 32 and
  // the 11 x 11 stride 4 first layer of an early image network, 3 -> 64 on 224 x 224, otherwise on the direct kernel).
  if (forced == 8 || forced < 0) {
    const int64_t need = padded_input_bytes(d->geom, s, forced == 8);
    tmq_conv2d_geom padded_geom = d->geom;
    padded_geom.IC = round_up(s.IC, 16);
    ConvShape padded_shape;
    const bool use = need > 0 && d->workspace != nullptr && d->workspace_bytes >= need && aligned(d->workspace, 16) &&
                     make_shape(&padded_geom, &padded_shape) == TMQ_OK;
    if (forced == 8 && !use) return TMQ_ERR_UNSUPPORTED;
    if (use) {
      const int64_t chunks = need / 16;
      enqueue(conv_pad_channels_kernel, dim3(static_cast<unsigned>(ceil_div(chunks, 256 * kPadBlocks))), dim3(256), 0, stream,
              static_cast<const uint8_t*>(d->x), static_cast<int>(s.IC), static_cast<int>(ceil_div(s.IC, 16)),
              static_cast<uint32_t>(chunks), s.B * s.H * s.W * s.IC, static_cast<uint8_t*>(d->workspace));
      if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
      tmq_conv2d_desc padded = *d;
      padded.x = d->workspace;
      padded.geom = padded_geom;
      padded.workspace = nullptr;
      padded.workspace_bytes = 0;
      padded.kernel = 0;
      padded.tile_rows = padded.tile_cols = 0;
      return run_conv<MODE>(&padded, post, out, stream);
    }
  }
  const bool mfma_ok = s.ICg % 16 == 0 && aligned(d->x, 16);
  if ((forced == 1 || forced == 2) && !mfma_ok) return TMQ_ERR_UNSUPPORTED;
  // pointwise layers over few input channels: pixels straight from memory against weights in registers
  {
    const bool rows_ok = pointwise_rows_ok(d->geom, s) && (MODE != kOutAcc32 || aligned(out, 4));
    if (forced == 9 && !rows_ok) return TMQ_ERR_UNSUPPORTED;
    if (forced == 9 || (forced < 0 && rows_ok && (pointwise_rows_first(s, po.any()) || !mfma_ok)))
      return launch_conv_pointwise_rows<MODE>(d, s, po, zp_f, lo_f, hi_f, out, stream);
  }
  // depthwise layers: four channels per lane on the vector ALU
  {
    // (32-bit byte offsets into the input and the output, also for the rows a window reaches past the image)
    const bool lanes_ok = s.taps_bytes > 0 && s.B * s.H * s.W * s.IC < (int64_t{1} << 31) &&
                          (s.H + s.KH * s.dh + s.sh + 8) * s.W * s.IC < (int64_t{1} << 31) &&
                          s.B * s.OH * s.OW * s.OC < (int64_t{1} << (MODE == kOutAcc32 ? 29 : 31)) && aligned(out, MODE == kOutAcc32 ? 4 : 1);
    if (forced == 7 && !lanes_ok) return TMQ_ERR_UNSUPPORTED;
    // Also where the groups would merge into 16-channel blocks for the matrix pipe, for the kernel sizes with a
    // register window (batch 32, against the merged groups on the halo tiles or the implicit GEMM: 3 x 3, 32
    // channels on 112 x 112 12.6 against 16.7 us; 96 channels, 112 x 112 -> 56 x 56: 13.9 against 25.2 us; 5 x 5, 240
    // channels on 28 x 28: 13.0 against 17.1 us; 7 x 7, 96 channels on 56 x 56: 22 against 72 us, 768 on 7 x 7: 6.7
    // against 242 us); other kernel sizes stay with the matrix pipe where they can.
    const bool lanes_first = s.KH == s.KW && (s.KH == 3 || s.KH == 5 || s.KH == 7);
    if (forced == 7 || (forced < 0 && lanes_ok && (!mfma_ok || lanes_first)))
      return launch_conv_depthwise<MODE>(d, s, po, zp_f, lo_f, hi_f, out, stream);
  }
  // channel counts (or an address) the 16-byte chunks of the kernels below cannot take:
  // kernel rows as runs of bytes where they are short enough
  if (forced == 4 || (forced < 0 && !mfma_ok)) {
    RunPlan rp;
    if (plan_runs(s, forced == 4 ? d->tile_rows : 0, &rp)) return launch_conv_runs<MODE>(d, s, rp, po, zp_f, lo_f, hi_f, out, stream);
    if (forced == 4) return TMQ_ERR_UNSUPPORTED;
  }
  if (!mfma_ok || forced == 3) {
    PlainArgs p{};
    p.x = static_cast<const uint8_t*>(d->x);
    p.w_packed = static_cast<const uint8_t*>(d->w_packed);
    p.colsum = d->w_colsum;
    p.w_scales = d->w_scales;
    p.bias = d->bias;
    p.w_scale_stride = d->w_per_channel ? 1 : 0;
    p.x_signed = d->x_signed;
    p.x_zp = d->x_zero_point;
    p.x_scale = d->x_scale;
    p.out_scale = d->out_scale;
    p.zp_f = zp_f; p.lo_f = lo_f; p.hi_f = hi_f;
    p.y = out;
    p.post = po;
    const int64_t blocks = ceil_div(rows * s.OC, 256);
    if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
    enqueue(conv_plain_kernel<MODE>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, s, p);
    return launch_status();
  }

  TilePlan plan;
  // (what needs no plan first: that takes the host 0.5 to 3 us)
  const bool tiles_ok = forced != 2 && !(forced < 0 && pointwise_gemm_first(s, po, 0)) &&
                        plan_tiles(s, forced == 1, d->tile_rows, d->tile_cols, &plan) &&
                        !(forced < 0 && pointwise_gemm_first(s, po, plan.rounds));
  if (forced == 1 && !tiles_ok) return TMQ_ERR_UNSUPPORTED;
  if (tiles_ok) {
    ConvTileArgs t{};
    t.x = static_cast<const uint8_t*>(d->x);
    t.w_packed = static_cast<const uint8_t*>(d->w_packed);
    t.colsum = d->w_colsum;
    t.w_scales = d->w_scales;
    t.bias = d->bias;
    t.y = out;
    t.w_kchunks = s.KC;
    t.group_bytes = s.group_bytes;
    t.H = static_cast<int>(s.H); t.W = static_cast<int>(s.W); t.IC = static_cast<int>(s.IC);
    t.OH = static_cast<int>(s.OH); t.OW = static_cast<int>(s.OW); t.OC = static_cast<int>(s.OC);
    t.KW = static_cast<int>(s.KW); t.icb = static_cast<int>(s.ICg / 16);
    t.kchunks = static_cast<int>(s.KH * s.KW * (s.ICg / 16));
    t.KS = plan.KS;
    t.sh = static_cast<int>(s.sh); t.sw = static_cast<int>(s.sw);
    t.ph = static_cast<int>(s.ph); t.pw = static_cast<int>(s.pw);
    t.dh = static_cast<int>(s.dh); t.dw = static_cast<int>(s.dw);
    t.ICg = static_cast<int>(s.ICg); t.OCg = static_cast<int>(s.OCg);
    t.n_tiles = static_cast<int>(ceil_div(s.OCg, kCtBN));
    t.TH = plan.TH; t.TW = plan.TW; t.HH = plan.HH; t.HW = plan.HW; t.pitch = plan.pitch;
    t.tiles_h = static_cast<int>(ceil_div(s.OH, plan.TH));
    t.tiles_w = static_cast<int>(ceil_div(s.OW, plan.TW));
    t.lds_x = plan.lds_x; t.lds_t = plan.lds_t; t.lds_tab = plan.lds_tab;
    t.through = MODE != kOutAcc32 && tiles_through(s, out) ? 1 : 0;
    t.w_scale_stride = d->w_per_channel ? 1 : 0;
    t.x_xor = d->x_signed ? 0u : 0x80808080u;
    t.pad_word = 0x01010101u * static_cast<uint32_t>(static_cast<uint8_t>(d->x_zero_point));
    t.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
    t.x_scale = d->x_scale;
    t.out_scale = d->out_scale;
    t.zp_f = zp_f; t.lo_f = lo_f; t.hi_f = hi_f;
    t.ri = plan.row_slots;
    t.rpp = kCtThreads / t.ri;
    t.cx = (plan.HH + t.rpp - 1) / t.rpp;
    t.xstep = static_cast<uint32_t>(t.rpp) * static_cast<uint32_t>(s.W) * static_cast<uint32_t>(s.IC);
    t.xdstep = t.rpp * t.ri * 16;
    t.post = po;
    t.rcp_tw = 1.0f / static_cast<float>(plan.TW);
    t.rcp_ri = 1.0f / static_cast<float>(t.ri);
    t.rcp_pslots = 16.0f / static_cast<float>(plan.pitch);
    t.rcp_icb = 1.0f / static_cast<float>(t.icb);
    t.rcp_kw = 1.0f / static_cast<float>(s.KW);
    return launch_conv_tiles<MODE>(s, plan, t, stream);
  }

  GemmArgs a{};
  XConvTable xs{};
  conv_gemm_operands(d, s, po, zp_f, lo_f, hi_f, out, &a, &xs);
  const bool table = conv_table_takes(s);
  const int64_t stages = ceil_div(s.Kp, kBK);
  ConvGemmTile tile = table ? conv_gemm_tile(rows, s.OCg, stages, po.any()) : conv_walk_tile(rows, s.OCg, stages);
  if (forced == 2 && !pinned_conv_tile(d->tile_rows, d->tile_cols, stages, &tile)) return TMQ_ERR_UNSUPPORTED;
  for (int64_t g = 0; g < s.groups; ++g) {
    a.w_packed = static_cast<const uint8_t*>(d->w_packed) + g * s.group_bytes;
    a.n_off = static_cast<int32_t>(g * s.OCg);
    xs.ic_off = static_cast<int>(g * s.ICg);
    rc = table ? launch_conv_gemm_tile<MODE>(tile, a, xs, stream) : launch_conv_gemm_walk<MODE>(tile, a, xs, stream);
    if (rc != TMQ_OK) return rc;
  }
  return TMQ_OK;
}

}  // namespace
}  // namespace tmq

using namespace tmq;

TMQ_EXPORT int64_t tmq_conv2d_packed_bytes(const tmq_conv2d_geom* g) {
  ConvShape s;
  if (make_shape(g, &s) != TMQ_OK) return 0;
  return s.groups * s.group_bytes + s.runs_bytes + s.taps_bytes;
}

TMQ_EXPORT int64_t tmq_conv2d_workspace_bytes(const tmq_conv2d_geom* g) {
  ConvShape s;
  if (make_shape(g, &s) != TMQ_OK) return 0;
  TilePlan tp;
  const int64_t need = patch_rows_bytes(*g, s, false);
  if (need > 0 && !(s.ICg % 16 == 0 && plan_tiles(s, false, 0, 0, &tp))) return need;
  return padded_input_bytes(*g, s, false);
}

TMQ_EXPORT int64_t tmq_conv2d_scratch_bytes(const tmq_conv2d_geom* g) {
  ConvShape s;
  return make_shape(g, &s) == TMQ_OK && conv_waves_tile(s, *g, false) != 0 ? 0 : tmq_conv2d_workspace_bytes(g);
}

TMQ_EXPORT int tmq_conv2d_out_hw(const tmq_conv2d_geom* g, int64_t* OH, int64_t* OW) {
  ConvShape s;
  const int rc = make_shape(g, &s);
  if (rc != TMQ_OK) return rc;
  if (OH != nullptr) *OH = s.OH;
  if (OW != nullptr) *OW = s.OW;
  return TMQ_OK;
}

TMQ_EXPORT int tmq_conv2d_prepack(const int8_t* w_ohwi, const tmq_conv2d_geom* g, void* packed,
                                  int32_t* colsum, tmq_stream_t stream) {
  ConvShape s;
  const int rc = make_shape(g, &s);
  if (rc != TMQ_OK) return rc;
  if (w_ohwi == nullptr || packed == nullptr || colsum == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(packed, 16)) return TMQ_ERR_ALIGNMENT;
  hipStream_t hs = as_stream(stream);
  const int64_t total = s.groups * s.group_bytes / 16;
  int64_t blocks = ceil_div(total, 256);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  enqueue(conv_prepack_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, hs,
          w_ohwi, s, total, static_cast<uint8_t*>(packed));
  if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  if (s.runs_bytes > 0) {
    const int64_t slots = s.runs_bytes / 16;
    enqueue(conv_prepack_runs_kernel, dim3(static_cast<unsigned>(ceil_div(slots, 256))), dim3(256), 0, hs,
            w_ohwi, s, slots, static_cast<uint8_t*>(packed) + s.runs_off);
    if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  }
  if (s.taps_bytes > 0) {
    enqueue(conv_prepack_taps_kernel, dim3(static_cast<unsigned>(ceil_div(s.taps_bytes, 256))), dim3(256), 0, hs,
            w_ohwi, s.IC, s.KH, s.KW, s.taps_bytes, static_cast<uint8_t*>(packed) + s.runs_off);
    if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  }
  blocks = ceil_div(s.OC, 256 / kWave);
  enqueue(conv_colsum_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, hs,
          w_ohwi, s.OC, s.KH * s.KW * s.ICgo, colsum);
  return launch_status();
}

TMQ_EXPORT int tmq_conv2d(const tmq_conv2d_desc* d, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  return d->out_signed ? run_conv<kOutS8>(d, nullptr, d->y, as_stream(stream))
                       : run_conv<kOutU8>(d, nullptr, d->y, as_stream(stream));
}

TMQ_EXPORT int tmq_conv2d_fused(const tmq_conv2d_desc* d, const tmq_conv2d_post* post,
                                tmq_stream_t stream) {
  if (d == nullptr || post == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  return d->out_signed ? run_conv<kOutS8>(d, post, d->y, as_stream(stream))
                       : run_conv<kOutU8>(d, post, d->y, as_stream(stream));
}

TMQ_EXPORT int tmq_conv2d_acc32(const tmq_conv2d_desc* d, int32_t* acc, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  return run_conv<kOutAcc32>(d, nullptr, acc, as_stream(stream));
}
