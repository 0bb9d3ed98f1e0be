// quantized::linear for gfx950: weight re-tiling, the MFMA GEMM dispatch, a
// weight-streaming kernel for decode-sized batches, and a plain kernel for
// shapes the vector paths do not take (K not a multiple of 16, unaligned rows).
#include <atomic>

#include "device_info.h"
#include "gemm_i8_core.h"
#include "gemm_i8_onepass.h"
#include "gemm_i8_persistent.h"
#include "gemm_i8_wring.h"
#include "gemm_i8_wloop.h"
#include "linear_dynamic_tiles.h"
#include "linear_resident.h"
#include "qparams.h"

// Layout that non-C++ bindings rely on (natural alignment, x86-64).
static_assert(sizeof(tmq_linear_desc) == 144, "tmq_linear_desc layout changed");
static_assert(sizeof(tmq_qparams) == 16, "tmq_qparams layout changed");

namespace tmq {
namespace {

constexpr int64_t kKPad = 128;  // packed k extent is a multiple of this

__host__ __device__ inline int64_t packed_kchunks(int64_t K) { return (K + kKPad - 1) / kKPad * (kKPad / 16); }

// ---------------------------------------------------------------------------
// prepack: one thread per 16-byte packed chunk (nb, kc, r)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void prepack_kernel(const int8_t* __restrict__ w, int64_t N,
                                                      int64_t K, int64_t ldw, int64_t KC,
                                                      int64_t total, bool vec,
                                                      uint8_t* __restrict__ packed) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= total) return;
  const int r = static_cast<int>(id & 15);
  const int64_t kc = (id >> 4) % KC;
  const int64_t nb = (id >> 4) / KC;
  const int64_t n = nb * 16 + r, k0 = kc * 16;
  v4i out = {0, 0, 0, 0};
  if (n < N && k0 < K) {
    const int8_t* src = w + n * ldw + k0;
    if (vec && k0 + 16 <= K) {
      out = ld16(src);
    } else {
      uint32_t words[4] = {0, 0, 0, 0};
      for (int b = 0; b < 16 && k0 + b < K; ++b)
        words[b >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(src[b])) << (8 * (b & 3));
      out = v4i{static_cast<int>(words[0]), static_cast<int>(words[1]), static_cast<int>(words[2]),
                static_cast<int>(words[3])};
    }
  }
  *reinterpret_cast<v4i*>(packed + id * 16) = out;
}

__global__ __launch_bounds__(256) void unpack_kernel(const uint8_t* __restrict__ packed, int64_t N,
                                                     int64_t K, int64_t ldw, int64_t KC,
                                                     int8_t* __restrict__ w) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= N * K) return;
  const int64_t n = id / K, k = id % K;
  w[n * ldw + k] = static_cast<int8_t>(packed[(((n >> 4) * KC + (k >> 4)) * 16 + (n & 15)) * 16 + (k & 15)]);
}

// colsum[n] = sum_k W[n][k]; one wavefront per weight row.
__global__ __launch_bounds__(256) void colsum_kernel(const int8_t* __restrict__ w, int64_t N,
                                                     int64_t K, int64_t ldw, bool vec,
                                                     int32_t* __restrict__ colsum) {
  const int lane = threadIdx.x % kWave;
  const int64_t n = static_cast<int64_t>(blockIdx.x) * (256 / kWave) + threadIdx.x / kWave;
  if (n >= N) return;
  const int8_t* row = w + n * ldw;
  int s = 0;
  int64_t k = 0;
  if (vec) {
    for (int64_t c = lane; c < K / 16; c += kWave) {
      const v4i v = ld16(row + c * 16);
      s = __builtin_amdgcn_sdot4(v.x, 0x01010101, s, false);
      s = __builtin_amdgcn_sdot4(v.y, 0x01010101, s, false);
      s = __builtin_amdgcn_sdot4(v.z, 0x01010101, s, false);
      s = __builtin_amdgcn_sdot4(v.w, 0x01010101, s, false);
    }
    k = K / 16 * 16;
  }
  for (int64_t i = k + lane; i < K; i += kWave) s += row[i];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
  if (lane == 0) colsum[n] = s;
}

// ---------------------------------------------------------------------------
// Decode-sized batches (M <= 16): the weight is read once, straight from HBM
// into MFMA operand registers (the packed layout is the 16x16x64 operand
// order), activations come from L2.  One block per 16 output channels, its
// eight waves split K and reduce through LDS.
//   D[i][j] of v_mfma_i32_16x16x64_i8: lane l, register r -> i = 4*(l/16)+r
//   (channel), j = l%16 (activation row).
// ---------------------------------------------------------------------------
constexpr int kDecodeWaves = 8;
constexpr int kDecodeMaxRows = 64;
constexpr int kDecodeRowsAuto = 16;  // up to here the automatic choice always streams the weights
// MG = groups of 16 activation rows (M <= 16 * MG): the weight operands are
// loaded once and multiplied with every group.
// ROWS = 4 (one group of at most four rows): a request for activations brings four k-blocks of the
// wave at once, so that a batch holds 8 registers of them instead of 32 and six waves fit a SIMD
// instead of five: 688 blocks (N = 11008) are then on the chip together instead of 512 and a rest
// (us, rows one to four, 16-row requests | these: K = 4096, N = 11008 11.2 | 9.6, N = 12288 12.5 | 10.3;
// K = 11008, N = 4096 9.8 | 9.1; K = 8192, N = 2048 6.9 | 6.0; K = 192, N = 8192 4.9 | 4.1; a kernel that only reads
// 45 MB takes 7.5).  Requests of two k-blocks for eight rows gain nothing (9.8 | 9.9).
//
// The 14 dwords in front of GemmArgs are everything the kernel's loads need.  The
// library is compiled with kernel-argument preloading, which hands up to 14
// leading scalar dwords of a kernel to its waves in SGPRs at launch, so the
// requests leave without waiting for a read of the argument buffer; the rest of
// the arguments is fetched under the weight stream.  The finishing threads'
// per-channel constants are requested first (cold, and memory serves requests
// in the order issued) and worked out under the first batch's requests, not behind its products; then each
// k-block's weights (HBM) and activations (L2).
// Measured at K = N = 4096 in a replayed graph of 40 cold weights: 5.25 us at
// M = 1, of which 1.9 us are what an empty kernel costs there, a kernel that
// only reads the 16.8 MB takes 4.1 us, and the one that also stores 4 KB of
// results 4.5 us (the store's acknowledgement ends the kernel); one or two
// accumulators and 4 / 8 / 16 waves all stay within 0.1 us.
// flags: bits 0-7 M, bit 8 per-channel weight scales, bit 9 unsigned activations.
// RAGGED: K (>= 16), the row pitch or the activation pointer is no multiple of 16.  The
// activation requests are the same 16 bytes per lane at whatever address the row has, the
// last chunk of a row is shifted into place; one launch instead of a pass that copies the rows onto
// the 16-byte grid first (that pass is what more rows take, and the vector path it then needs).
template <int MODE, int MG, bool RAGGED = false, int ROWS = 16>
__global__ __launch_bounds__(kDecodeWaves* kWave, ROWS == 4 ? 6 : 1) void linear_decode_kernel(
    const uint8_t* __restrict__ w_packed, const uint8_t* __restrict__ x, const int32_t* __restrict__ colsum,
    const float* __restrict__ w_scales, const float* __restrict__ bias, int32_t K, int32_t ldx, int32_t N,
    uint32_t flags, GemmArgs a) {
  constexpr int kWaves = kDecodeWaves;
  constexpr int kBatch = 8;  // 64-byte k-blocks in flight per wave: 64 KB of weights per block
  constexpr int kSpan = 16 / ROWS;  // k-blocks whose activations one request brings
  static_assert(MG == 1 || ROWS == 16, "fewer than 16 rows: one group");
  static_assert(kBatch % kSpan == 0, "whole requests");
  // The eight waves' partial sums meet in one [4 registers][64 lanes] array per row group:
  // every wave adds its accumulators with LDS atomics as it finishes (a wave instruction covers
  // 64 consecutive words: no bank conflicts, and the early waves' additions are off the block's
  // critical path), and the 64 finishing threads read four words each instead of 32.
  __shared__ int s_sum[MG][4][kWave];
  const int t = threadIdx.x, lane = t % kWave, wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int lr = lane & 15, lc = lane >> 4;
  const int nb = blockIdx.x;
  const int M = static_cast<int>(flags & 0xffu);
  for (int i = t; i < MG * 4 * kWave; i += kWaves * kWave) (&s_sum[0][0][0])[i] = 0;
  // (before any global request is made: the barrier's wait for outstanding memory
  // operations is then a wait for this one LDS store)
  __syncthreads();
  const int KB = (K + 63) >> 6;
  // The 64 threads that finish a block: thread -> activation row within a
  // group, channel group of 4.
  const int fm = t >> 2, fg = t & 3;
  int c_cs[4] = {0, 0, 0, 0};
  float c_ws[4] = {1.f, 1.f, 1.f, 1.f}, c_b[4] = {0.f, 0.f, 0.f, 0.f};
  if (t < 64) {
    const int ws_stride = (flags >> 8) & 1;
    const float* const bsrc = bias != nullptr ? bias : w_scales;  // a load that always has an address
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = nb * 16 + 4 * fg + j;
      const int np = n < N ? n : 0;
      c_cs[j] = colsum[np];
      if (MODE != kOutAcc32) {
        c_ws[j] = w_scales[np * ws_stride];
        c_b[j] = bsrc[bias != nullptr ? np : 0];  // (looked at in `constants`: a select here would wait for it)
      }
    }
  }
  const uint8_t* wp = w_packed + static_cast<int64_t>(nb) * (packed_kchunks(K) * 256) + lc * 256 + lr * 16;
  // Activations are loaded with four consecutive lanes on the 64 bytes one row
  // contributes to a k-block (lane -> row lane / 4, 16-byte piece lane % 4): a
  // quad of lanes then asks for one cache line instead of four.  With at most ROWS < 16 rows
  // the other lanes take the same rows of the wave's next k-blocks.  The multiply
  // wants row lane % 16 and piece lane / 16, so every loaded register goes
  // through cross-lane permutations (for k-block i of a request, lane l takes from lane
  // 4 (ROWS i + l % ROWS) + l / 16; rows ROWS ... 15 repeat others and are not stored).
  const int sr = (lane >> 2) & (ROWS - 1), sp = lane & 3, sk = lane / (4 * ROWS);
  const int perm_addr = (4 * (lr & (ROWS - 1)) + lc) * 4;
  bool xrow[MG];
  const uint8_t* xp[MG];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg) {
    xrow[mg] = mg * 16 + sr < M;
    xp[mg] = x + static_cast<int64_t>(xrow[mg] ? mg * 16 + sr : 0) * ldx;  // the row's first byte: always readable
  }
  const int xor_word = (flags >> 9) & 1 ? static_cast<int>(0x80808080u) : 0;
  const v4i xmask = {xor_word, xor_word, xor_word, xor_word};
  // This lane's 16-byte piece of k-block kb of its row; `ok`: the piece has bytes of the row.
  auto piece = [&](const uint8_t* row, int kb, bool ok) {
    const int at = ok ? kb * 64 + sp * 16 : 0;
    if constexpr (RAGGED) return ld16_any(row + (at <= K - 16 ? at : K - 16));
    else return ld16(row + at);
  };
  // (behind the load, in the k-block that ends the row)
  auto settle = [&](v4i v, int kb) {
    if constexpr (RAGGED) {
      const int over = kb * 64 + sp * 16 - (K - 16);
      return over > 0 && over < 16 ? shift_down_bytes(v, over) : v;
    }
    return v;
  };
  // Two accumulators per row group, used in turn: a multiply-accumulate does not
  // wait for the one before it.
  v4i acc2[MG][2];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg) acc2[mg][0] = acc2[mg][1] = v4i{0, 0, 0, 0};
  // Every load of a batch is unconditional (addresses clamped into the operands,
  // the activation operand of a block that does not exist set to zero after the
  // load), so that the counts of outstanding loads are exact and the k-blocks are
  // multiplied one by one as they arrive; with a load under a condition the
  // compiler waits for all of them before the first product.
  // `meanwhile` runs under the latency of the requests.
  auto batch = [&](int kb0, auto meanwhile) {
    constexpr int kReq = kBatch / kSpan;  // activation requests per row group
    v4i wf[kBatch], xf[MG][kReq];
    bool xok[MG][kReq];
    const auto request_x = [&](int mg, int q) {
      const int kb = kb0 + (q * kSpan + sk) * kWaves;
      xok[mg][q] = kb < KB && xrow[mg] && (kb * 64 + sp * 16 < K);
      xf[mg][q] = piece(xp[mg], kb, xok[mg][q]);
    };
    // Requests are counted back in the order issued.  With one group of 16 rows the weights
    // (memory, the critical path) go first, each followed by its activations; with more
    // groups, or where a request serves several k-blocks, the activations (L2) all go first, so that their
    // cross-lane permutations run while the weights are still on their way (K = N = 4096: M = 1 5.25 against 5.46 us
    // the other way round, M = 32 7.5 against 7.8 us).
    constexpr bool kFirst = MG >= 2 || kSpan > 1;
    if constexpr (kFirst) {
#pragma unroll
      for (int q = 0; q < kReq; ++q)
#pragma unroll
        for (int mg = 0; mg < MG; ++mg) request_x(mg, q);
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int kb = kb0 + u * kWaves;
      const int kbc = kb < KB ? kb : KB - 1;
      wf[u] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wp + static_cast<int64_t>(kbc) * 1024));
      if constexpr (!kFirst) request_x(0, u);
    }
    meanwhile();
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int mg = 0; mg < MG; ++mg) {
        const int q = u / kSpan;
        if (u % kSpan == 0) {
          v4i xw = xf[mg][q];
          // (the k-block that ends the rows: the same for the whole wave with one k-block per request)
          if (RAGGED && kb0 + (u + kSpan - 1) * kWaves >= KB - 1) xw = settle(xw, kb0 + (u + sk) * kWaves);
          xf[mg][q] = xok[mg][q] ? (xw ^ xmask) : v4i{0, 0, 0, 0};
        }
        v4i xv;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          xv[c] = __builtin_amdgcn_ds_bpermute(perm_addr + (u % kSpan) * (16 * ROWS), xf[mg][q][c]);
        acc2[mg][u & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[u], xv, acc2[mg][u & 1], 0, 0, 0);
      }
  };
  // requantisation constants, by the wave that finishes the block, under its first requests
  v4f bdiv = {0.f, 0.f, 0.f, 0.f}, mult = {0.f, 0.f, 0.f, 0.f};
  float bmul = 1.f;
  int acc0[4] = {0, 0, 0, 0};
  auto constants = [&]() {
    if (wave != 0) return;
    const XQuant xq = x_quant(a);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc0[j] = xq.coef * c_cs[j];
      if (MODE == kOutF32) {
        mult[j] = xq.scale * c_ws[j];
        bdiv[j] = a.bias != nullptr ? c_b[j] : 0.f;
      } else if (MODE != kOutAcc32) {
        const float atw = xq.scale * c_ws[j];
        mult[j] = atw / a.out_scale;
        bdiv[j] = a.bias != nullptr ? bias_term(a.w_scale_stride == 0, c_b[j], atw) : 0.f;
        bmul = bias_mul(a.w_scale_stride == 0, atw);  // (per tensor: the same for every j)
      }
    }
  };
  // (two copies of the batch: with the constants inside the loop the registers of one copy hold fewer waves)
  if (wave < KB) batch(wave, constants);  // (K >= 1: wave 0 has a k-block)
  for (int kb0 = wave + kWaves * kBatch; kb0 < KB; kb0 += kWaves * kBatch) batch(kb0, []() {});
  v4i acc[MG];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg) acc[mg] = acc2[mg][0] + acc2[mg][1];
#pragma unroll
  for (int mg = 0; mg < MG; ++mg)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __hip_atomic_fetch_add(&s_sum[mg][r][lane], acc[mg][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __syncthreads();
  if (t < 64) {
    const int g = fg;
#pragma unroll
    for (int mg = 0; mg < MG; ++mg) {
      const int64_t m = mg * 16 + fm;
      if (m >= a.M) continue;
      int raw[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)  // channel 4 g + j of row fm: register j of lane 16 g + fm
        raw[j] = s_sum[mg][j][16 * g + fm] + acc0[j];
      const int64_t n = nb * 16 + 4 * g;
      if (MODE == kOutAcc32) {
        int32_t* dst = static_cast<int32_t*>(a.y) + m * a.ldy + n;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < a.N) dst[j] = raw[j];
      } else if (MODE == kOutF32) {
        store_f32x4(a, m, n, raw, mult, bdiv);
      } else {
        const uint32_t packed = requant4<MODE>(raw, bdiv, bmul, mult, a.zp_f, a.lo_f, a.hi_f);
        uint8_t* dst = static_cast<uint8_t*>(a.y) + m * a.ldy + n;
        if (n + 3 < a.N && (a.ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 3) == 0) {
          *reinterpret_cast<uint32_t*>(dst) = packed;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (n + j < a.N) dst[j] = static_cast<uint8_t>(packed >> (8 * j));
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Dynamically quantized linear for a handful of rows (M <= 16, M * K <= 16384),
// float in, float out, one launch.  The weight-streaming kernel above with the
// activation quantization inside: every block requests its weights, then reads
// the whole float input (at most 64 KB, from L2), reduces min / max, derives the
// parameters (ChooseQuantizationParams, one thread), quantizes the values it
// holds into LDS -- product and zero point rounded once, as PyTorch's CPU
// quantized::linear_dynamic does while packing -- and multiplies from there.
// Every block repeats the same few microseconds of work on the input, under the
// latency of its own weight stream, instead of waiting for a launch that does
// it once.  Same arithmetic, same results as the two launches.
// ---------------------------------------------------------------------------
constexpr int64_t kDynSmallMaxValues = 16384;
// kHeld: float4 groups of the input per thread, M * K / 4 <= kHeld * 512 (a template
// parameter: the loads are unconditional so that the load counter stays exact).
template <int kHeld>
__global__ __launch_bounds__(kDecodeWaves* kWave) void linear_decode_dynamic_kernel(
    GemmArgs a, const float* __restrict__ x, int64_t ldxf, int reduce_range) {
  constexpr int kWaves = kDecodeWaves;
  constexpr int kBatch = 8;
  static_assert(kHeld * 4 * kWaves * kWave <= kDynSmallMaxValues, "held values");
  extern __shared__ __attribute__((aligned(16))) uint8_t sx[];  // [M][pitch] activation codes
  __shared__ int s_sum[4][kWave];  // the waves' partial sums, added with LDS atomics (see linear_decode_kernel)
  __shared__ float s_range[2 * kWaves + 3];
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  const int lr = lane & 15, lc = lane >> 4;
  const int64_t nb = blockIdx.x;
  const int64_t KB = ceil_div(a.K, 64);
  const int K = static_cast<int>(a.K);
  const int pitch = (K + 15) / 16 * 16 + 16;  // rows 16 bytes apart in the banks
  const uint8_t* wp = a.w_packed + nb * a.w_kchunks * 256 + lc * 256 + lr * 16;
  // per-channel constants of the 64 finishing threads, requested first
  const int fm = t >> 2, fg = t & 3;
  int c_cs[4] = {0, 0, 0, 0};
  float c_ws[4] = {1.f, 1.f, 1.f, 1.f}, c_b[4] = {0.f, 0.f, 0.f, 0.f};
  if (t < 64) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = nb * 16 + 4 * fg + j;
      const int64_t np = n < a.N ? n : 0;
      c_cs[j] = a.colsum[np];
      c_ws[j] = a.w_scales[np * a.w_scale_stride];
      if (a.bias != nullptr) c_b[j] = a.bias[np];
    }
  }
  // ---- the input: requested first (loads return in order: behind the weight
  // stream it would arrive only after it), held in registers between the range
  // pass and the quantization
  HeldRows<kHeld, kWaves * kWave> rows;
  rows.load(x, ldxf, static_cast<int>(a.M), K, t);
  // then the first batch of weights: on its way while the input is processed
  v4i wf[kBatch];
#pragma unroll
  for (int u = 0; u < kBatch; ++u) {
    const int64_t kb = wave + u * kWaves;
    const int64_t kbc = kb < KB ? kb : KB - 1;
    wf[u] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wp + kbc * 1024));
  }
  __builtin_amdgcn_sched_barrier(0);
  if (t < 4 * kWave) (&s_sum[0][0])[t] = 0;  // (two barriers before the first addition)
  float mn = __builtin_inff(), mx = -__builtin_inff();
  rows.range(mn, mx);
  float scale, inv, zp_f;
  block_qparams<kWaves>(mn, mx, s_range, t, reduce_range != 0, [] { __syncthreads(); }, scale, inv, zp_f);
  rows.codes(inv, zp_f, [&](int row, int c4, uint32_t q) { *reinterpret_cast<uint32_t*>(sx + row * pitch + c4 * 4) = q; });
  __syncthreads();
  // ---- the product, activation operands from LDS (rows past M are zero)
  const v4i xmask = {static_cast<int>(0x80808080u), static_cast<int>(0x80808080u), static_cast<int>(0x80808080u),
                     static_cast<int>(0x80808080u)};
  const bool xrow = lr < a.M;
  const uint8_t* xp = sx + (xrow ? lr : 0) * pitch + lc * 16;
  v4i acc = {0, 0, 0, 0};
  for (int64_t kb0 = wave; kb0 < KB; kb0 += kWaves * kBatch) {
    if (kb0 != wave) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int64_t kb = kb0 + u * kWaves;
        wf[u] = kb < KB ? __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wp + kb * 1024)) : v4i{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t kb = kb0 + u * kWaves;
      const bool xok = kb < KB && xrow && (kb * 64 + lc * 16 < a.K);
      // (bytes of LDS past the end of a row meet the zeros the packed weights end in;
      // weights of a block past K were loaded from a clamped address: the zero
      // activation operand removes them from the sum, x ^ 0x80 alone would not)
      const v4i xf = xok ? ld16(xp + kb * 64) ^ xmask : v4i{0, 0, 0, 0};
      const v4i wv = kb < KB ? wf[u] : v4i{0, 0, 0, 0};
      acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv, xf, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    __hip_atomic_fetch_add(&s_sum[r][lane], acc[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  v4f mult = {0.f, 0.f, 0.f, 0.f}, bias = {0.f, 0.f, 0.f, 0.f};
  int acc0[4] = {0, 0, 0, 0};
  if (t < 64) {
    const int coef = 128 - static_cast<int>(zp_f);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc0[j] = coef * c_cs[j];
      mult[j] = scale * c_ws[j];
      bias[j] = c_b[j];
    }
  }
  __syncthreads();
  if (t < 64 && fm < a.M) {
    int raw[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) raw[j] = s_sum[j][16 * fg + fm] + acc0[j];
    store_f32x4(a, fm, nb * 16 + 4 * fg, raw, mult, bias);
  }
}

// ---------------------------------------------------------------------------
// Activation rows onto the 16-byte grid: K bytes at any address and pitch -> `chunks`
// 16-byte chunks, zeros past K.  The copy that lets every vector kernel run a product whose
// K or pointer is off that grid: M x K bytes in and out (the product reads them many times
// over), against the plain kernel's byte-wise loop, which is all such products had: 517 rows
// quantized, through 1000 -> 2051 -> 1000 features and dequantized: 4014 -> 27 us.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void regrid_rows_kernel(const uint8_t* __restrict__ x, int64_t ldx, int32_t K,
                                                          uint32_t chunks, uint32_t total, v4i* __restrict__ out) {
  const uint32_t id = blockIdx.x * 256 + threadIdx.x;
  if (id >= total) return;
  const uint32_t row = id / chunks;
  const int k0 = static_cast<int>(id - row * chunks) * 16;
  const uint8_t* src = x + static_cast<int64_t>(row) * ldx;
  v4i v = {0, 0, 0, 0};
  if (K >= 16) {
    const int at = k0 <= K - 16 ? k0 : K - 16;
    v = shift_down_bytes(ld16_any(src + at), k0 - at);
  } else {
    uint32_t w[4] = {0, 0, 0, 0};
    for (int b = 0; b < K; ++b) w[b >> 2] |= static_cast<uint32_t>(src[b]) << (8 * (b & 3));
    v = v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])};
  }
  out[id] = v;
}

// ---------------------------------------------------------------------------
// Plain kernel: any K, any alignment, no scratch memory.  One thread per (m, group of 4 channels).
// ---------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256) void linear_plain_kernel(GemmArgs a, XLinear xs, int x_signed) {
  const int64_t groups = ceil_div(a.N, 4);
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= a.M * groups) return;
  const int64_t m = id / groups, n = (id % groups) * 4;
  const uint8_t* xr = xs.x + m * xs.ldx;
  int raw[4] = {0, 0, 0, 0};
  for (int64_t k = 0; k < a.K; ++k) {
    const int xv = x_signed ? static_cast<int>(static_cast<int8_t>(xr[k])) : static_cast<int>(xr[k]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t nn = n + j;  // rows past N are zero in the packed buffer's last block
      const int wv = static_cast<int8_t>(
          a.w_packed[(((nn >> 4) * a.w_kchunks + (k >> 4)) * 16 + (nn & 15)) * 16 + (k & 15)]);
      raw[j] += xv * wv;
    }
  }
  v4f bdiv, mult;
  float bmul = 1.f;
  const XQuant xq = x_quant(a);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t np = n + j < a.N ? n + j : 0;
    // plain accumulation used the true activation value, so only -x_zp*colsum is left
    raw[j] += xq.coef * a.colsum[np];
    if (MODE == kOutF32) {
      mult[j] = xq.scale * a.w_scales[np * a.w_scale_stride];
      bdiv[j] = a.bias != nullptr ? a.bias[np] : 0.f;
    } else if (MODE != kOutAcc32) {
      const float atw = xq.scale * a.w_scales[np * a.w_scale_stride];
      mult[j] = atw / a.out_scale;
      bdiv[j] = a.bias != nullptr ? bias_term(a.w_scale_stride == 0, a.bias[np], atw) : 0.f;
      bmul = bias_mul(a.w_scale_stride == 0, atw);
    }
  }
  if (MODE == kOutAcc32) {
    int32_t* dst = static_cast<int32_t*>(a.y) + m * a.ldy + n;
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N) dst[j] = raw[j];
  } else if (MODE == kOutF32) {
    store_f32x4(a, m, n, raw, mult, bdiv);
  } else {
    const uint32_t packed = requant4<MODE>(raw, bdiv, bmul, mult, a.zp_f, a.lo_f, a.hi_f);
    uint8_t* dst = static_cast<uint8_t*>(a.y) + m * a.ldy + n;
    for (int j = 0; j < 4; ++j)
      if (n + j < a.N) dst[j] = static_cast<uint8_t>(packed >> (8 * j));
  }
}

template <int BM, int BN, int WM, int WN, int MODE, int PD = 4, bool WDMA = false, int KW = 1, bool XWIDE = false,
          bool THROUGH = true, class XSRC = XLinear>
int launch_gemm(const GemmArgs& a, const XSRC& xs, hipStream_t s) {
  const int64_t blocks = ceil_div(a.M, BM) * ceil_div(a.N, BN);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  if (ceil_div(a.K, kBK) < KW) return TMQ_ERR_UNSUPPORTED;  // a stage for every wave group
  enqueue(gemm_i8_kernel<BM, BN, WM, WN, MODE, XSRC, PD, WDMA, KW, XWIDE, THROUGH>,
          dim3(static_cast<unsigned>(blocks)), dim3(WM * WN * KW * kWave), 0, s, a, xs);
  return launch_status();
}
// Tiles that are chosen for outputs of any size (the others run a round or a few of them, 13 MB at most).
template <int BM, int BN, int WM, int WN, int MODE, int PD = 4, bool WDMA = false, bool XWIDE = false>
int launch_gemm_any_size(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  if constexpr (MODE == kOutU8 || MODE == kOutS8) {
    if (!bytes_through(a)) return launch_gemm<BM, BN, WM, WN, MODE, PD, WDMA, 1, XWIDE, false>(a, xs, s);
  }
  return launch_gemm<BM, BN, WM, WN, MODE, PD, WDMA, 1, XWIDE>(a, xs, s);
}

// 64 x 64 (64 x 128) tiles with all of K in LDS (K <= 1024; the caller checked the address ranges).
template <int MODE, int BN = 64>
int launch_gemm_onepass(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  const int64_t tiles_m = ceil_div(a.M, 64), tiles_n = ceil_div(a.N, BN);
  if (tiles_n > 0x7fffffff || tiles_m > 65535) return TMQ_ERR_UNSUPPORTED;
  enqueue(gemm_i8_onepass_kernel<MODE, BN>,
          dim3(static_cast<unsigned>(tiles_n), static_cast<unsigned>(tiles_m)), dim3(BN * 4), 0, s, a, xs);
  return launch_status();
}

// Whether the XCDs take runs of a small grid's tiles (tile_of_block): several row tiles over 900 KB of weights and more that
// the grid's order would spread over the XCDs (us, weights from memory, without | with: 129 x 656 -> 3040 5.7 | 4.7, 137 x 688 ->
// 2272 5.3 | 4.7, 70 x 1280 -> 5184 7.3 | 6.3, 1129 x 3072 -> 448 8.6 | 7.8; 277 x 704 -> 640 3.8 | 4.2).
bool tile_runs(int64_t tiles_m, int64_t tiles_n, const GemmArgs& a) {
  return tiles_m > 1 && tiles_n % 8 != 0 && a.N * a.K >= 900 * 1024;
}

// 32 x 32 tiles whose four waves split K (K <= 1024; the caller checked the address ranges).
template <int MODE>
int launch_gemm_ksplit(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  const int64_t tiles_m = ceil_div(a.M, 32), tiles_n = ceil_div(a.N, 32);
  if (tiles_n > 0x7fffffff || tiles_m > 65535 || a.K > kOnePassMaxK) return TMQ_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>(tiles_n), static_cast<unsigned>(tiles_m));
  if (tiles_n * tiles_m <= 0x7fffffff && tile_runs(tiles_m, tiles_n, a))
    enqueue(gemm_i8_ksplit_kernel<MODE, true>, grid, dim3(256), 0, s, a, xs);
  else
    enqueue(gemm_i8_ksplit_kernel<MODE, false>, grid, dim3(256), 0, s, a, xs);
  return launch_status();
}

// 64 x 64 tiles whose eight waves split K, weights through registers, activations through
// a ring per wave (K <= 4096; the caller checked the address ranges).
template <int MODE>
int launch_gemm_wring(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  const int64_t tiles_m = ceil_div(a.M, 64), tiles_n = ceil_div(a.N, 64);
  if (tiles_n > 0x7fffffff || tiles_m > 65535 || a.K > kWringMaxK || a.K % 16 != 0) return TMQ_ERR_UNSUPPORTED;
  enqueue(gemm_i8_wring_kernel<MODE>,
          dim3(static_cast<unsigned>(tiles_n), static_cast<unsigned>(tiles_m)), dim3(kWringThreads), 0, s, a, xs);
  return launch_status();
}

// Tiles of 32 rows x 32 or 64 channels whose waves split K and walk their shares in pieces (the caller checked the
// address ranges).
template <int MODE>
int launch_gemm_wloop(const GemmArgs& a, const XLinear& xs, bool wide, hipStream_t s) {
  const int64_t tiles_m = ceil_div(a.M, 32), tiles_n = ceil_div(a.N, wide ? 64 : 32);
  if (tiles_n * tiles_m > 0x7fffffff || tiles_m > 65535) return TMQ_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>(tiles_n), static_cast<unsigned>(tiles_m)), block(kWloopWaves * kWave);
  if (wide) enqueue(gemm_i8_wloop_kernel<MODE, 2>, grid, block, 0, s, a, xs);
  else enqueue(gemm_i8_wloop_kernel<MODE, 1>, grid, block, 0, s, a, xs);
  return launch_status();
}
// ... and for rows off the 16-byte grid.
template <int MODE>
int launch_gemm_wloop_ragged(const GemmArgs& a, const XLinear& xs, bool wide, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(ceil_div(a.N, wide ? 64 : 32)), static_cast<unsigned>(ceil_div(a.M, 32)));
  const XLinearRagged rows{xs.x, xs.ldx};
  if (wide) enqueue(gemm_i8_wloop_kernel<MODE, 2, XLinearRagged>, grid, dim3(kWloopWaves * kWave), 0, s, a, rows);
  else enqueue(gemm_i8_wloop_kernel<MODE, 1, XLinearRagged>, grid, dim3(kWloopWaves * kWave), 0, s, a, rows);
  return launch_status();
}

// The same for K up to 4096 (cfg 25, 26), two tiles of 32 channels side by side in a block where one round holds those only
// (us, weights from memory, four waves a tile and two blocks a CU | pairs: 71 x 1120 -> 3200 5.6 | 4.6, 1445 x 1472 -> 288 7.4 |
// 5.3, 512 x 2048 -> 1024 6.7 | 6.1).
bool wstream_pairs(int64_t M, int64_t N) {
  return ceil_div(M, 32) * ceil_div(N, 32) > 256 && ceil_div(M, 32) * ceil_div(N, 64) <= 256;
}

// One block per CU walks the 256 x 256 tiles (byte or float outputs, direct copies two
// stages wide: the caller checked their address and K ranges).
template <int MODE>
int launch_gemm_persistent(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  if constexpr (MODE == kOutU8 || MODE == kOutS8 || MODE == kOutF32) {
    const int64_t tiles = ceil_div(a.M, 256) * ceil_div(a.N, 256);
    const int cus = cu_count();
    if (cus < 8 || tiles > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
    // several rounds: a multiple of 8 blocks, so that the tile sequence deals
    // every XCD its own run of tiles
    const int64_t grid = tiles <= cus ? tiles : cus / 8 * 8;
    const dim3 blocks(static_cast<unsigned>(grid)), threads(kPersistThreads);
    // Whole lines leave past the L2s at any size, beside the next tile's products (us without | with: 4096 x 1024 -> 4096 23.2 |
    // 21.3, 4096 x 11008 -> 4096 149.5 | 147.7, 4096 x 512 -> 11008 45 MB 42.7 | 37.7; 112 shapes of 6 to 120 MB 7 % ahead,
    // none behind); parts of lines as for the other tiles (173660 x 768 -> 144 25 MB 46.6 | 52.2).
    if constexpr (MODE != kOutF32) {
      if (!whole_lines(a) && !bytes_through(a)) {
        enqueue(gemm_i8_persistent_kernel<MODE, false>, blocks, threads, 0, s, a, xs);
        return launch_status();
      }
    }
    enqueue(gemm_i8_persistent_kernel<MODE, true>, blocks, threads, 0, s, a, xs);
    return launch_status();
  } else {
    return TMQ_ERR_UNSUPPORTED;
  }
}

// Scratch for activation rows that are off the 16-byte grid (regrid_rows_kernel).
int64_t regrid_pitch(int64_t K) { return round_up(K, 16); }
int64_t regrid_bytes(int64_t M, int64_t K) { return round_up(M * regrid_pitch(K), 256); }
// (the copy's index arithmetic is 32 bits wide: up to 32 GiB of activations)
bool regrid_limits_ok(int64_t M, int64_t K) { return K > 0 && K <= 0x7fffff00 && M * (regrid_pitch(K) / 16) <= 0x7fffff00; }
int launch_regrid(const XLinear& xs, int64_t M, int64_t K, void* out, hipStream_t s) {
  const int64_t chunks = regrid_pitch(K) / 16, total = M * chunks;
  enqueue(regrid_rows_kernel, dim3(static_cast<unsigned>(ceil_div(total, 256))), dim3(256), 0, s,
          xs.x, xs.ldx, static_cast<int32_t>(K), static_cast<uint32_t>(chunks), static_cast<uint32_t>(total),
          static_cast<v4i*>(out));
  return launch_status();
}

// Weight streaming for up to 16 rows that are off the 16-byte grid.
template <int MODE>
int launch_linear_decode_ragged(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  const uint32_t flags = static_cast<uint32_t>(a.M) | (a.w_scale_stride != 0 ? 0x100u : 0u) |
                         (a.x_xor != 0 ? 0x200u : 0u);
  const auto launch = [&](auto rows_tag) {
    enqueue(linear_decode_kernel<MODE, 1, true, decltype(rows_tag)::value>,
            dim3(static_cast<unsigned>(ceil_div(a.N, 16))), dim3(kDecodeWaves * kWave), 0, s,
            a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, static_cast<int32_t>(a.K), static_cast<int32_t>(xs.ldx),
            static_cast<int32_t>(a.N), flags, a);
  };
  if (a.M <= 4) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 16>{});
  return launch_status();
}

// Weight streaming for up to 64 rows: one block per 16 channels.
template <int MODE>
int launch_linear_decode(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  // (the kernel derives the packed pitch from K, as prepack does)
  if (a.w_kchunks != packed_kchunks(a.K)) return TMQ_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>(ceil_div(a.N, 16))), block(kDecodeWaves * kWave);
  const int32_t k32 = static_cast<int32_t>(a.K), ldx32 = static_cast<int32_t>(xs.ldx);
  const int32_t n32 = static_cast<int32_t>(a.N);
  const uint32_t flags = static_cast<uint32_t>(a.M) | (a.w_scale_stride != 0 ? 0x100u : 0u) |
                         (a.x_xor != 0 ? 0x200u : 0u);
  switch ((a.M + 15) / 16) {
    case 1:
      if (a.M <= 4)
        enqueue(linear_decode_kernel<MODE, 1, false, 4>, grid, block, 0, s,
                a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, k32, ldx32, n32, flags, a);
      else
        enqueue(linear_decode_kernel<MODE, 1>, grid, block, 0, s,
                a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, k32, ldx32, n32, flags, a);
      break;
    case 2: enqueue(linear_decode_kernel<MODE, 2>, grid, block, 0, s,
            a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, k32, ldx32, n32, flags, a); break;
    case 3: enqueue(linear_decode_kernel<MODE, 3>, grid, block, 0, s,
            a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, k32, ldx32, n32, flags, a); break;
    default: enqueue(linear_decode_kernel<MODE, 4>, grid, block, 0, s,
            a.w_packed, xs.x, a.colsum, a.w_scales, a.bias, k32, ldx32, n32, flags, a); break;
  }
  return launch_status();
}

// Up to 64 rows whose activations (16 MG x K bytes, MG = groups of 16 rows) fit the
// kernel's LDS area: one block per CU streams the channel groups it owns.
bool resident_limits_ok(int64_t M, int64_t N, int64_t K, int64_t ldx, int cus) {
  if (M < 1 || M > 64 || K < 64 || K % 16 != 0 || cus < 1) return false;
  const int64_t mg = ceil_div(M, 16), groups = ceil_div(N, 16);
  return 16 * mg * ceil_div(K, 64 * kResidentWaves) * (64 * kResidentWaves) <= kResidentXBytes && groups <= static_cast<int64_t>(kResidentMaxGroups) * cus &&
         N <= 0x7ffffff0 && ldx <= (int64_t{1} << 40);
}

// Two blocks of eight waves per CU where the rows fit half the LDS area (one group of rows,
// K <= 4096) and a block still owns at most 32 channel groups: the two blocks' bursts of
// requests interleave (M = 8, K = 4096, N = 32000: 25.2 -> 24.0 us; N = 16384, K = 1024: 6.7 -> 6.0 us;
// N = 8192, K = 2048: 6.2 -> 5.8 us).  Not below two groups per block at K > 2048: the rows are then
// staged twice per CU for nothing (N = 5120, K = 4096, M = 16: 7.7 -> 8.8 us; N = 11008: 10.6 -> 11.0 us).
bool resident_pair(int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t groups = ceil_div(N, 16);
  return M <= 16 && 16 * ceil_div(K, 64 * 8) * (64 * 8) <= kResidentXBytes / 2 && groups <= int64_t{32} * 2 * cus &&
         groups >= (K <= 2048 ? 2 : 4) * static_cast<int64_t>(cus);
}

template <int MODE>
int launch_linear_resident(const GemmArgs& a, const XLinear& xs, hipStream_t s) {
  const int cus = cu_count();
  if (!resident_limits_ok(a.M, a.N, a.K, xs.ldx, cus)) return TMQ_ERR_UNSUPPORTED;
  const int64_t groups = ceil_div(a.N, 16);
  if (resident_pair(a.M, a.N, a.K, cus)) {
    const dim3 grid(static_cast<unsigned>(groups < 2 * cus ? groups : 2 * cus)), block(8 * kWave);
    enqueue(linear_resident_kernel<MODE, 1, 8>, grid, block, 0, s, a, xs, nullptr, 0, 0);
    return launch_status();
  }
  const dim3 grid(static_cast<unsigned>(groups < cus ? groups : cus)), block(kResidentThreads);
  switch ((a.M + 15) / 16) {
    case 1: enqueue(linear_resident_kernel<MODE, 1>, grid, block, 0, s, a, xs, nullptr, 0, 0); break;
    case 2: enqueue(linear_resident_kernel<MODE, 2>, grid, block, 0, s, a, xs, nullptr, 0, 0); break;
    case 3: enqueue(linear_resident_kernel<MODE, 3>, grid, block, 0, s, a, xs, nullptr, 0, 0); break;
    default: enqueue(linear_resident_kernel<MODE, 4>, grid, block, 0, s, a, xs, nullptr, 0, 0); break;
  }
  return launch_status();
}

// ---- split K for a few hundred rows against a long K.  The tile grid of such a
// product is far smaller than the chip (M = 128, N = 4096: 32 tiles of
// 128 x 128) and every block walks all of K alone at the latency of one stage
// after the other, so K is cut into `splits` runs of whole stages: splits x
// tiles blocks write raw int32 partial sums [split][M][ldp] into a caller-owned
// workspace and a second kernel adds them up and requantises.  Writing and
// re-reading the partial sums costs about 10 us at these sizes, which the
// shorter k loops repay from K = 8192 on (measured: M = 128, N = 4096,
// K = 11008: 38.5 -> 25 us; K = 4096: 14.6 -> 20 us, hence no split there).
struct SplitPlan {
  int splits = 1;   // 1: single launch
  int stages = 0;   // k stages (64 bytes of K) per split
  int64_t ldp = 0;  // row pitch of a partial-sum slice, int32 elements
};

constexpr int64_t kSplitBlocks = 256;    // blocks wanted: one per CU
constexpr int64_t kSplitMinKT = 128;     // shortest k loop (stages) worth cutting
constexpr int64_t kSplitMinStages = 16;  // shortest run of stages per split

// ---- 17 ... 64 rows: several kernels can run such a product, and which is fastest
// depends on the shape.  Estimated microseconds per launch, fitted to sweeps with
// cold weights (more weight sets in rotation than the last-level cache holds):
//  * the weight-streaming kernel: a block of 16 channels streams its K x 16 weight
//    bytes once and re-reads the activations of every group of 16 rows, so one round
//    of blocks (N <= 4096) costs a base that grows with the weight bytes plus a share
//    per row group that grows with K (K = N = 4096: 6.4 / 7.5 / 11.3 us at M = 17 / 32 / 64;
//    N = 4096, K = 8192: 10.2 / 12.2 / 18.8 us), and further rounds cost about three
//    quarters of the first (N = K = 8192, two rounds: 19.2 / 20.9 / 34.8 us; N = 11008,
//    K = 4096, three rounds: 15.1 / 16.3 / 28.1 us);
//  * 64 x 64 tiles walk K at the latency of one stage after the other, almost
//    whatever M is (K = N = 4096 with two wave groups: 12.6 / 14.3 us at
//    M = 32 / 64; N = 11008: 14.6 / 16.9 us), and K <= 1024 fits LDS whole
//    (gemm_i8_onepass.h: K = 1024 on 32 x 32 tiles: 3.8 / 4.1 / 4.9 us at N = 1024 / 4096 / 8192);
//  * split K moves the weights at about 4.5 TB/s plus 10 us for the partial sums
//    (N = 4096, K = 11008: 21.7 us at M = 64 against 27.0 us streaming; K = 8192, M = 48:
//    18.0 against 15.5 us streaming).
enum class SmallRows { kStream, kTiles, kSplit };

// 64 x 64 tiles whose k loop two wave groups share: at most one block per CU and a loop long enough to
// pay for adding the groups' sums (us, one group | two: K = 6592, N = 1600, M = 266 21.3 | 16.2; K = 4160,
// N = 4096, M = 256 14.8 | 12.2; K = 2064, N = 1000, M = 517 9.0 | 8.1; K = 1536, N = 2048, M = 300 7.4 | 6.7;
// K = 1344, N = 168, M = 2017 7.1 | 6.7; K = 1088, N = 1024, M = 200 5.9 | 5.9; 275 tiles, K = 1600 9.8 | 10.2;
// four groups are behind two at all of these).
bool two_wave_groups_fit(int64_t M, int64_t N, int64_t K) {
  return ceil_div(M, 64) * ceil_div(N, 64) <= 256 && ceil_div(K, kBK) >= 20;
}

SplitPlan plan_split_tiles(int64_t M, int64_t N, int64_t K);

// Shapes for the tiles of 32 rows whose waves split K and stream their weights through
// registers (gemm_i8_wloop.h): K beyond what the kernels with all operands in LDS take, one round of blocks of 32 or 64
// channels.  With more than that it loses to the larger tiles.  Returns the channels per tile: 32 (K <= 2048: by pairs
// where single ones are more than a round, wstream_pairs), 64; 0: neither.
int wstream_tile(int64_t M, int64_t N, int64_t K) {
  if (K <= kOnePassMaxK || K > 4096) return 0;
  const bool pairs = ceil_div(M, 32) * ceil_div(N, 64) <= 256;
  if (ceil_div(M, 32) * ceil_div(N, 32) <= 256 || (K <= 2048 && pairs)) return 32;
  return pairs ? 64 : 0;
}

// One round of 64 x 64 tiles against K > 4096 whose last row tile is at least three
// quarters full, up to 128 rows: the kernel that copies K through LDS in phases takes the
// same time whatever the rows (N = K = 5120: 17.1 ... 17.9 us from 40 to 128 rows; N = K = 8192:
// 26.5 us at 64 rows), while two wave groups slow down as the tiles fill (20.9 us and 29.3 us
// at 64 rows; N = 4096, K = 11008, M = 64: 32.2 against 37.3 us).  With a tile half empty, or
// from 192 rows on, the wave groups are ahead (N = 4096, K = 14336, M = 256: 42.4 against 45.6 us).
// (K = 4096 against N >= 10240, where the tiles of 32 rows no longer fit one round: M = 64, N = 11008: 16.2 against
// 17.5 us; N = 14336: 17.3 against 18.1 us; at 128 rows the wave groups are ahead, N = 8192: 15.7 against 16.2 us)
bool phased_ring_preferred(int64_t M, int64_t N, int64_t K) {
  if (K % 16 != 0 || ceil_div(M, 64) * ceil_div(N, 64) > 256 || (M - 1) % 64 < 47) return false;
  return K > 4096 ? M <= 128 : (K == 4096 && M <= 64 && N >= 10240);
}

// More than 32 rows against K beyond 4096, one round of tiles of 32 rows: eight waves a tile that walk K in pieces
// (gemm_i8_wloop.h).  Us, the best other kernel | it, weights from memory:
//   up to 256 tiles of 32 x 32: 63 x 5376 -> 107 11.5 | 7.35; 49 x 4160 -> 430 9.9 | 6.35; 76 x 9168 -> 2336 17.8 | 12.0; 37 x 4624 -> 304
//     8.9 | 6.3; 135 x 11552 -> 1488 21.1 | 13.5;
//   up to 256 of 32 x 64: 71 x 5936 -> 3504 16.0 | 12.0; 127 x 4576 -> 4080 15.7 | 10.8; 42 x 6704 -> 6624 19.4 | 14.4; 74 x 8752 -> 5040
//     21.7 | 16.8; 65 x 10496 -> 4880 22.8 | 17.9; 85 x 11296 -> 2736 21.2 | 20.6;
//   up to 32 rows weights stream as fast (18 x 5296 -> 1584 7.2 | 8.3, 26 x 8144 -> 192 8.0 | 8.8; 30 x 4656 -> 128 6.9 | 6.1), up to
//     40 against more than 17 Mi weights short of K = 10240 likewise when that line was drawn (now ahead, 36 x 6288 -> 5632 17.7 | 12.9).
// The tiles that walk K as a ring of phases keep their shapes up to K = 5632 and, of 64 channels, those of more than 32 Mi weights,
// which their tests hold as the automatic choice; measured, this kernel is ahead there throughout (128 x 4608 -> 256 14.7 | 6.6,
// 48 x 4288 -> 5024 15.0 | 10.3).  Measured up to K = 12288.  Returns the channels per tile, 0: not such a shape.
constexpr int64_t kWloopMaxK = 12288, kWloopRingMinK = 5632;
int wloop_tile(int64_t M, int64_t N, int64_t K) {
  if (M <= 32 || K <= 4096 || K > kWloopMaxK || K % 16 != 0) return 0;
  if (M <= 40 && N * K > int64_t{17} << 20 && K < 10240) return 0;
  const bool ring = phased_ring_preferred(M, N, K);
  if (ring && K < kWloopRingMinK) return 0;
  if (ceil_div(M, 32) * ceil_div(N, 32) <= 256) return 32;
  return ceil_div(M, 32) * ceil_div(N, 64) <= 256 && !(ring && N * K > int64_t{32} << 20) ? 64 : 0;
}

// (`tiles` beyond K = 1024 prices one round as two wave groups and the ring of phases: the lone tiles' ring that runs now is
// up to a tenth faster, and the kernel in pieces is not priced here at all)
SmallRows small_rows_path(int64_t M, int64_t N, int64_t K, bool workspace) {
  // Where the tiles of 32 rows with the weights through registers fit, they are measured directly against the
  // weight-streaming kernel, which keeps K > 3008 up to 32 rows (two row groups) while its blocks fit one round (us, tiles |
  // streaming: 18 x 2176 -> 545 4.4 | 5.0, 28 x 2288 -> 2000 4.5 | 5.1, 20 x 2576 -> 144 4.4 | 4.8, 32 x 3024 -> 544 level at 5.0,
  // 29 x 3744 -> 160 5.5 | 5.0, 24 x 3696 -> 2661 7.2 | 5.9, 31 x 4096 -> 1600 6.1 | 5.4; 24 x 2784 -> 4864 6.4 | 8.9).
  if (wstream_tile(M, N, K) != 0)
    return K > 3008 && M <= 32 && N <= 4096 ? SmallRows::kStream : SmallRows::kTiles;
  const double mib = static_cast<double>(N) * static_cast<double>(K) / 1048576.0;
  const double stages = static_cast<double>(ceil_div(K, kBK));
  const double rows = static_cast<double>(M);
  const double kk = static_cast<double>(K) / 1024.0;
  const double stream_rounds = static_cast<double>(ceil_div(ceil_div(N, 16), 256));
  const double round_mib = static_cast<double>(std::min<int64_t>(N, 4096)) * static_cast<double>(K) / 1048576.0;
  const double one_round = 1.9 + 0.09 * round_mib + static_cast<double>(ceil_div(M, 16)) * std::max(1.6, 0.42 * kk);
  const double stream = stream_rounds <= 1.0 ? one_round : one_round * (0.3 + 0.75 * stream_rounds);
  const double nblk = static_cast<double>(ceil_div(M, 64) * ceil_div(N, 64));
  double tiles;
  if (K <= kOnePassMaxK && K > 256 && ceil_div(M, 32) * ceil_div(N, 32) <= 512)
    // all of K in LDS, 32 x 32 tiles (K = 1024: 3.8 / 3.8 / 4.1 / 4.9 us at N = 1024 / 2048 / 4096 / 8192;
    // more than 256 tiles, N = 8192, M = 40: 5.4 us)
    tiles = 3.6 + 0.13 * mib + (ceil_div(M, 32) * ceil_div(N, 32) > 256 ? 0.5 : 0.0);
  else if (K <= kOnePassMaxK && nblk <= 256.0)  // 64 x 64 tiles (K = N = 1024: 5.6 us, N = 1024, K = 256: 3.1 us)
    tiles = 2.0 + 3.8 * kk + 0.012 * std::max(0.0, nblk - 64.0);
  else if (phased_ring_preferred(M, N, K))
    // (N = 4096: 25.3 / 32.2 / 40.9 us at K = 8192 / 11008 / 14336; N = K = 5120: 17.4 us; N = K = 8192: 26.5 us)
    tiles = 3.3 + 2.65 * kk + 0.2 * std::max(0.0, static_cast<double>(N) - 4096.0) / 1024.0;
  else if (two_wave_groups_fit(M, N, K))
    tiles = (4.4 + 0.123 * stages + 0.013 * std::max(0.0, nblk - 64.0)) *
            (1.0 + 0.35 * (rows / 64.0) * (rows / 64.0) * std::min(1.0, stages / 172.0));
  else
    tiles = (3.0 + 0.2 * stages) * (1.0 + nblk / 1024.0);
  const double best = std::min(stream, tiles);
  if (workspace && plan_split_tiles(M, N, K).splits > 1) {
    // (N = 4096: 18.0 / 21.3 / 23.5 us at K = 8192 / 11008 / 14336, 48 rows)
    const double split = 10.0 + 0.23 * mib + 0.025 * rows;
    if (split < best) return SmallRows::kSplit;
  }
  return stream <= tiles ? SmallRows::kStream : SmallRows::kTiles;
}

SplitPlan plan_split_tiles(int64_t M, int64_t N, int64_t K) {
  SplitPlan p;
  if (M <= kDecodeRowsAuto || K % 16 != 0) return p;
  const int64_t KT = ceil_div(K, kBK);
  const int64_t tiles = ceil_div(M, 128) * ceil_div(N, 128);
  if (KT < kSplitMinKT || tiles > kSplitBlocks / 2) return p;
  int64_t splits = kSplitBlocks / tiles;
  if (splits > KT / kSplitMinStages) splits = KT / kSplitMinStages;
  if (splits < 2) return p;
  const int64_t stages = ceil_div(KT, splits);
  splits = ceil_div(KT, stages);
  // a last run of fewer than six stages (one turn of the direct-copy ring) is
  // merged into the split before it: the kernel's last split multiplies
  // everything from (splits - 1) * stages to the end of K
  if (KT - (splits - 1) * stages < 6) --splits;
  if (splits < 2) return p;
  p.splits = static_cast<int>(splits);
  p.stages = static_cast<int>(stages);
  p.ldp = (N + 3) / 4 * 4;
  return p;
}

// Bytes and floats are not split where one round holds the product in 64 x 64 tiles but not in tiles of 32 rows: the lone tiles' ring is ahead up to
// K = 10752, and beyond against more than 550 thousand outputs (us, split | ring, weights from memory: 661 x 8544 -> 1408 28.4 |
// 21.1, 478 x 8736 -> 1152 25.9 | 21.3, 168 x 8656 -> 4736 27.2 | 23.3, 1110 x 11504 -> 794 33.7 | 27.2, 683 x 11872 -> 832 27.8 |
// 28.8; 194 x 10976 -> 2560 23.2 | 26.0, 180 x 13024 -> 2752 26.8 | 34.7, 80 x 12896 -> 5632 27.0 | 31.0).  The split stays where
// it would go to the ring of phases (split | phases | lone ring: 128 x 10960 -> 7038 34.5 | 35.6 | 35.9, 114 x 10576 -> 4815 26.2 |
// 32.1 | 31.1, 119 x 9056 -> 6172 27.2 | 29.0 | 28.1, 123 x 13184 -> 7505 35.7 | 40.6 | 40.1, 128 x 8240 -> 4200 23.4 | 26.5 | 26.7).
bool ring_ahead_of_split(int64_t M, int64_t N, int64_t K) {
  return ceil_div(M, 64) * ceil_div(N, 64) <= 256 && ceil_div(M, 32) * ceil_div(N, 64) > 256 && (K < 10752 || M * N > 550000) &&
         !phased_ring_preferred(M, N, K);
}

// The plan the automatic choice follows: none for the rows that stream the
// weights, and for 17 ... 64 rows only where the estimate above prefers it.
SplitPlan plan_split(int64_t M, int64_t N, int64_t K) {
  if (M > kDecodeRowsAuto && M <= kDecodeMaxRows && small_rows_path(M, N, K, true) != SmallRows::kSplit)
    return SplitPlan{};
  return plan_split_tiles(M, N, K);
}

int64_t split_workspace_bytes(const SplitPlan& p, int64_t M) {
  return p.splits > 1 ? p.splits * M * p.ldp * static_cast<int64_t>(sizeof(int32_t)) : 0;
}

// Second kernel of a split-K product: a block owns 256 consecutive channels and
// `rows` rows.  Its threads first compute the 256 channels' constants, one
// channel each, into LDS (the two divisions per channel would otherwise be
// repeated by every row); then a thread adds the `splits` partial sums of four
// consecutive channels of one row at a time and runs the epilogue of the
// single-launch kernels (same helper, same operation order).
template <int MODE>
__global__ __launch_bounds__(256) void splitk_finish_kernel(GemmArgs a, const int32_t* parts, int splits,
                                                            int64_t ldp, int64_t slice, int rows) {
  __shared__ __attribute__((aligned(16))) int s_add[256];
  __shared__ __attribute__((aligned(16))) float s_mult[256];
  __shared__ __attribute__((aligned(16))) float s_bdiv[256];
  const int t = threadIdx.x;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * 256;
  {
    const XQuant xq = x_quant(a);
    const int64_t nj = n0 + t < a.N ? n0 + t : a.N - 1;
    float mult = 0.f, bdiv = 0.f;
    if (MODE != kOutAcc32) {
      const float atw = xq.scale * a.w_scales[nj * a.w_scale_stride];
      if (MODE == kOutF32) {
        mult = atw;
        bdiv = a.bias != nullptr ? a.bias[nj] : 0.f;
      } else {
        mult = atw / a.out_scale;
        bdiv = a.bias != nullptr ? bias_term(a.w_scale_stride == 0, a.bias[nj], atw) : 0.f;
      }
    }
    s_add[t] = xq.coef * a.colsum[nj];
    s_mult[t] = mult;
    s_bdiv[t] = bdiv;
  }
  __syncthreads();
  const int q = t & 63;
  const int64_t n = n0 + q * 4;
  if (n >= a.N) return;
  const v4i add = *reinterpret_cast<const v4i*>(&s_add[q * 4]);
  const v4f mult = *reinterpret_cast<const v4f*>(&s_mult[q * 4]);
  const v4f bdiv = *reinterpret_cast<const v4f*>(&s_bdiv[q * 4]);
  const bool plain_u8 = MODE == kOutU8 && a.lo_f <= 0.f && a.hi_f >= 255.f;
  const float bmul = (MODE == kOutU8 || MODE == kOutS8)
                         ? bias_mul(a.w_scale_stride == 0, x_quant(a).scale * a.w_scales[0]) : 1.0f;
  const int64_t mbeg = static_cast<int64_t>(blockIdx.y) * rows;
  const int64_t mend = mbeg + rows < a.M ? mbeg + rows : a.M;
  for (int64_t m = mbeg + (t >> 6); m < mend; m += 4) {
    const int32_t* src = parts + m * ldp + n;
    v4i sum = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(src));
    for (int sp = 1; sp < splits; ++sp)
      sum += __builtin_nontemporal_load(reinterpret_cast<const v4i*>(src + sp * slice));
    sum += add;
    const int raw[4] = {sum.x, sum.y, sum.z, sum.w};
    if constexpr (MODE == kOutAcc32) {
      int32_t* dst = static_cast<int32_t*>(a.y) + m * a.ldy + n;
      for (int j = 0; j < 4; ++j)
        if (n + j < a.N) dst[j] = raw[j];
    } else if constexpr (MODE == kOutF32) {
      store_f32x4(a, m, n, raw, mult, bdiv);
    } else {
      const uint32_t q4 = plain_u8 ? requant4<MODE, false>(raw, bdiv, bmul, mult, a.zp_f, a.lo_f, a.hi_f)
                                   : requant4<MODE, true>(raw, bdiv, bmul, mult, a.zp_f, a.lo_f, a.hi_f);
      uint8_t* dst = static_cast<uint8_t*>(a.y) + m * a.ldy + n;
      if (n + 3 < a.N && (reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
        *reinterpret_cast<uint32_t*>(dst) = q4;
      } else {
        for (int j = 0; j < 4; ++j)
          if (n + j < a.N) dst[j] = static_cast<uint8_t>(q4 >> (8 * j));
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int PD = 4, bool WDMA = false, bool XWIDE = false>
int launch_gemm_split(const GemmArgs& a, const XLinear& xs, const SplitPlan& p, hipStream_t s) {
  const int64_t blocks = ceil_div(a.M, BM) * ceil_div(a.N, BN);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  enqueue(gemm_i8_kernel<BM, BN, WM, WN, kOutAcc32, XLinear, PD, WDMA, 1, XWIDE>,
          dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(p.splits)), dim3(WM * WN * kWave), 0, s, a, xs);
  return launch_status();
}

template <int MODE>
int run_split(const GemmArgs& a, const XLinear& xs, const SplitPlan& p, void* workspace, bool dma_ok,
              hipStream_t s) {
  GemmArgs part = a;  // first kernel: pure sums of (x ^ flip) * w, no zero-point term
  part.acc_coef = 0;
  part.acc_base = 0;
  part.f_kind = TMQ_FLOAT_F32;  // (32-bit words whatever kind of float the second kernel writes)
  part.x_qp_dev = nullptr;
  part.y = workspace;
  part.ldy = p.ldp;
  part.splits = p.splits;
  part.split_stages = p.stages;
  part.split_stride = a.M * p.ldp;
  const int rc = dma_ok ? launch_gemm_split<128, 128, 2, 2, 3, true, true>(part, xs, p, s)
                        : launch_gemm_split<128, 128, 2, 2>(part, xs, p, s);
  if (rc != TMQ_OK) return rc;
  // rows per block: enough blocks to hide the loads' latency, then longer runs
  const int rows = a.M <= 256 ? 4 : 16;
  const int64_t bx = ceil_div(a.N, 256), by = ceil_div(a.M, rows);
  if (bx > 0x7fffffff || by > 65535) return TMQ_ERR_UNSUPPORTED;  // a split product has a few hundred rows
  enqueue(splitk_finish_kernel<MODE>, dim3(static_cast<unsigned>(bx), static_cast<unsigned>(by)), dim3(256), 0, s,
          a, static_cast<const int32_t*>(workspace), p.splits, p.ldp, a.M * p.ldp, rows);
  return launch_status();
}

// ---- which kernel runs a product: a host-side function of the shape alone, so that
// it can be queried (tmq_linear_kernel_choice) and swept without a device.
struct LinearQuery {
  int64_t M, N, K, ldx;
  int64_t n_off = 0;
  int mode = kOutU8;             // EpilogueMode
  bool vec_ok = true;            // K, the row pitch and the activation pointer are multiples of 16
  bool workspace_attached = false;
  int64_t workspace_bytes = 0;   // usable (16-byte aligned) split-K scratch
};
// cfg: tmq_linear_desc::kernel - 1.  0-7, 14, 17, 19, 22, 23: tiles of gemm_i8_kernel (1, 2, 6, 7, 17, 19: copied straight
// into LDS where K and the pitch allow it); 8: weight
// streaming; 9: plain kernel; 13: split K (plan in `split`); 20: persistent 256 x 256 tiles;
// 21 / 24: all of K in LDS (64 x 64 / 32 x 32 tiles); 25 / 26: weights through registers
// (32 x 32 / 32 x 64 tiles); 27: the same with 64 x 64 tiles and the activations in a ring
// per wave; 28: activations resident in LDS, one block per CU streams its channel groups; 29 / 30: tiles of 32 rows x 32 / 64
// channels whose waves walk their shares of K in pieces;
// kNoKernel: the forced kernel does not take this shape.
constexpr int kNoKernel = -2;
struct LinearChoice {
  int cfg = kNoKernel;
  int groups = 1;  // wave groups that share the k loop of a 64 x 64 tile (cfg 2; cfg 14 always has two)
  bool onepass = false;  // 64 x 128 tiles with all of K in LDS (cfg 23)
  SplitPlan split;
};

// Limits of the kernels' own index arithmetic, shared by the choice and the launches.
// Direct-copy kernels: 256 rows of either operand addressed with 32-bit offsets, and
// their three-stage ring runs at least once around.
bool dma_limits_ok(int64_t K, int64_t ldx) { return ldx <= (int64_t{1} << 23) && K <= (int64_t{1} << 23) && K > 2 * kBK; }
// The copies two stages wide walk K in runs of six stages.
bool wide_limits_ok(int64_t K, int64_t ldx) { return dma_limits_ok(K, ldx) && K > 5 * kBK; }
// All of K in LDS / weights through registers: 32-bit offsets over 64 rows of either
// operand, N * 4 as a 32-bit offset.
bool onepass_limits_ok(const LinearQuery& q) {
  return q.K % 16 == 0 && q.K <= (int64_t{1} << 23) && q.ldx <= (int64_t{1} << 23) && q.N + q.n_off < (int64_t{1} << 29);
}
// The weight-streaming kernel takes K, the row pitch and N as 32-bit arguments.
bool stream_limits_ok(const LinearQuery& q) {
  return q.M <= kDecodeMaxRows && ceil_div(q.N, 16) <= 0x7fffffff && q.K <= 0x7fffff00 && q.ldx <= 0x7fffffff &&
         q.N <= 0x7ffffff0;
}

// Where the kernel that keeps the activations in LDS is ahead of a block per 16 channels
// (cold weights, us, resident | streaming; neither depends on N beyond what is shown):
//   K <= 2048, from N = 2048 on, any M <= 16:  K = N = 2048: 4.0 ... 4.2 | 4.2 ... 4.7;  N = 4096, K = 1024: 3.9 | 4.2 ... 4.5;  N = 8192, K = 1024:
//     4.8 ... 5.0 | 5.8 ... 6.3;  N = 4096, K = 2048: 4.5 | 4.7 ... 5.0;  N = 65536, K = 2048: 24.5 | 35 ... 42
//   longer K, 14 rows and more (the streaming blocks re-read the rows from the L2s), from N = 5120 on:
//     K = 4096, M = 16: N = 5120 7.7 | 8.6, N = 11008 10.6 | 12.3, N = 32000 25.4 | 32.2, N = 128256 97 | 122;
//     N = K = 8192, M = 16: 14.7 | 16.1  (M = 12: N = 5120 7.6 | 7.8, N = 8192 9.1 | 8.6: one full round of
//     streaming blocks, two per CU, is that kernel's best case)
//   5 ... 13 rows at K = 4096 beyond that round, N >= 10240: M = 8: N = 11008 10.8 | 11.3 ... 12.2, N = 32000
//     24.0 | 25.6, N = 128256 91.7 | 95.7;  M = 12: N = 49152 38.2 | 39.6, N = 65536 50.3 | 54.4
//   (fewer rows: level up to N = 32000, then the independent blocks stream faster: N = 128256, M = 1: 89 | 85;
//   N = 4096 at K >= 4096: level or behind, 6.1 | 5.9 at M = 16)
//   a K that leaves the streaming blocks a short last pass (K = N = 5120: 8.4 ... 8.7 | 9.2 ... 11.3 at M = 1 ... 12)
//   17 ... 32 rows: a narrow band between the tiles of 32 rows, which no longer fit one round, and the 64 x 128
//   tiles (K = 4096, M = 24 / 32: N = 11008 11.9 / 12.2 against 12.5 / 12.7 us, N = 16384 15.5 / 15.7 against
//   16.4 / 16.7 us; N = 8192: level with 32 x 32 tiles; N = 32000: 26.6 against 24.5 us for 64 x 128 tiles).
bool resident_preferred(const LinearQuery& q) {
  if (!q.vec_ok || q.K < 1024 || q.M > 32 || !resident_limits_ok(q.M, q.N, q.K, q.ldx, 256)) return false;
  if (q.M > 16) return q.K > 2048 && q.N >= 10240 && q.N <= 20480;
  if (q.K <= 2048) return q.N >= 2048;
  if (q.K > 4096 && q.K % 4096 != 0 && q.K % 4096 <= 2048 && q.N >= 5120) return true;
  return (q.M >= 14 && q.N >= 5120) || (q.M >= 5 && q.N >= 10240);
}

// Five rows and more against the very largest N at K > 2048: the pipelined 64 x 128 tiles, mostly padding
// in their rows, stream such a weight faster than either kernel above -- two and more long-running blocks
// per CU, each with its own ring of stages (cold weights, K = 4096, us, tiles | rows resident | a block per 16
// channels: N = 128256: M = 16 85.0 | 93.5 | 118, M = 8 87.3 | 93.5 | 97.2, M = 1 87.4 | 88 | 85.0;
// N = 65536: M = 16 47.6 | 51.4 | 63.8, M = 8 47.6 | 48.9 | 51.2; below, the resident rows are ahead:
// N = 49152, M = 16: 40.1 | 38.7; N = 32000: 26.8 | 25.8; at K = 2048 the two are level up to N = 128256).
bool huge_n_tiles_preferred(const LinearQuery& q) {
  return q.vec_ok && q.M >= 5 && q.M <= 16 && q.K > 2048 && q.N >= 65536;
}

// The one-launch dynamic linear: which of its two kernels, where both take the shape.  The block per CU
// that quantizes the rows once is ahead almost everywhere (cold weights, us, it | a block per 16 channels
// each quantizing the rows: K = N = 4096, M = 4: 7.7 | 8.1; N = 11008, M = 4: 12.3 | 15.2; N = 32000, M = 4:
// 26.3 | 35.2; N = 4096, K = 1024, M = 16: 6.1 | 7.0; N = 16384, K = 1024, M = 1: 6.7 | 10.3; N = 4096,
// K = 8192, M = 1: 9.8 | 10.1), except one or two rows against a single round of blocks at K = 4096
// (K = N = 4096, M = 1: 6.6 | 6.1).
bool dynamic_resident_preferred(int64_t M, int64_t N, int64_t K) {
  return !(M <= 2 && N <= 4096 && K > 2048 && K <= 4096);
}

// 64 x 128 tiles with all of K in LDS, where 64 x 64 ones would need a second round of blocks and these fit
// one, up to K = 256 (beyond, tile_by_rounds finds better ones; raw accumulators keep them; us, these | the pipelined tiles: K = 768, N = 3072: M = 384 5.8 | 6.6, M = 512 5.8 | 6.7, M = 640 5.9 | 6.8;
// K = 256, N = 2000, M = 1000 4.3 | 5.6; K = 64, N = 1000, M = 2000 4.7 | 6.7; K = 512, N = 1024, M = 2048 5.1 | 6.1;
// two rounds of them, K = 640, N = 1500, M = 1500: 10.4 | 8.2).  A K of four phases waits for the ring once:
// K = 1024: N = 1024, M = 2048 (512 tiles of 64 x 64) 6.9 | 7.5, N = 300, M = 4096 (320) 7.2 | 7.7, N = 1600,
// M = 700 (275) 7.8 | 7.3; K = 1008, N = 2051, M = 517 (297) 8.4 | 7.5.
bool onepass_wide_preferred(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ceil_div(M, 64) * ceil_div(N, 64);
  return K <= kOnePassMaxK && tiles > (K <= 768 ? 256 : 300) && ceil_div(M, 64) * ceil_div(N, 128) <= 256;
}

// Tiles of products over K <= kRoundsMaxK by the time their rounds take (us, u = tiles / 256 CUs, st = stages of 64 k-bytes):
//   start + round max(floor, by_u u) + full rounds of `on_cu` tiles per CU at fill + rate st each, start holding the fill of
// the last one: per_u u and max(floor, rate0 + rate1 u) st.  The constants are fitted to shapes drawn over M = 24 .. 110000,
// N = 64 .. 12288 and K = 64 .. 3600 (weights in the cache of the memory side; mean error 5 to 7 %), because the thresholds
// below, fitted to few sizes, miss by a tenth between those.  On 43 shapes with K from 64 to 3584 and weights from memory the
// tile they name is 1.5 % behind the best of all kernels on average, 17 % at most (M = 783, N = 1856, K = 3584 19.5 against
// 16.7 us for 128 x 64; M = 8000, N = 1000, K = 128 9.5 | 8.1 for 64 x 128).  Gained (us): M = 603, N = 2304, K = 768 6.1 -> 5.3 (64 x 64 copies for 64 x 128 with all of K in LDS);
// M = 642, N = 2304, K = 1920 12.1 -> 8.6, M = 2417, N = 832, K = 1344 9.4 -> 7.8 (for 128 x 128); M = 1690, N = 2616,
// K = 112 8.3 -> 6.5 (64 x 64 for 128 x 128 by registers); weights from memory, M = 460, N = 1728, K = 960 8.0 -> 6.0.
struct TileRate {
  int cfg, bm, bn;
  double on_cu, start, per_u, floor, rate0, rate1, fill, full;
};
constexpr int64_t kRoundsMaxK = 3600;
// A lone 64 x 64 tile on a CU has room for a ring of six stages: nothing where its weights come from a cache, but from
// memory M = 131, N = 3845, K = 2128 13.3 -> 9.5 us and M = 176, N = 2880, K = 2496 14.7 -> 10.9 (eight stages: 9.6 and 11.0).
bool one_round_ring(int64_t M, int64_t N, int64_t K) {
  return ceil_div(M, 64) * ceil_div(N, 64) <= 256 && K > 5 * kBK;
}
constexpr TileRate kShortRates[] = {
    // one or two stages: register staging
    {2, 64, 64, 6, 3.27, 0.47, 0.19, 0.0, 0.106, 3.14, 0.57},
    {3, 256, 256, 1, 6.11, 2.59, 0.81, 0.0, 1.05, 6.14, 0.82},
};
constexpr TileRate kRates[] = {
    // three and more: direct copies (2: 64 x 64, 1 / 7: 128 x 128 with copies of one / two stages)
    {2, 64, 64, 4, 3.14, 0.305, 0.116, 0.0, 0.119, 1.72, 0.45},
    {1, 128, 128, 1, 4.28, 0.66, 0.181, 0.138, 0.164, 1.40, 0.274},
    {7, 128, 128, 1, 4.51, 0.85, 0.177, 0.146, 0.128, 2.03, 0.238},
    {17, 128, 256, 1, 4.44, 1.97, 0.327, 0.0, 0.470, 2.67, 0.428},
    {6, 256, 256, 1, 7.35, 1.37, 0.489, 0.274, 0.601, 6.94, 0.767},
};
// Tiles of 64 x 128 and 128 x 64, copied straight into a ring of six stages where one round of them has a block per CU:
// a lone block's three stages in registers are what it waits for (us, registers | ring: M = 641, N = 1600, K = 8064 32.1 |
// 24.5; M = 133, N = 9984, K = 11776 52.0 | 42.1; M = 440, N = 2752, K = 3136 13.7 | 11.7; M = 514, N = 2432, K = 7104 128 x 64
// 29.0 | 23.7).  128 x 64 is two thirds activations, whose copies of 64 bytes touch two lines each off the 64-byte grid:
// no gain there (M = 261, N = 3712, K = 5200 23.0 | 24.2; M = 189, N = 6656, K = 4080 18.8 | 19.0).
bool oblong_ring(int64_t M, int64_t N, int64_t K, int64_t ldx, int bm, int bn) {
  return ceil_div(M, bm) * ceil_div(N, bn) <= 256 && K > 5 * kBK && dma_limits_ok(K, ldx) && (bm == 64 || K % kBK == 0);
}
// ... and taken there from K = 1280 on, where 64 x 64 tiles are more than a round (us, the choice before | 64 x 128 in a
// ring: M = 1829, N = 800, K = 1552 9.9 | 8.3; M = 875, N = 1600, K = 1680 10.8 | 8.8; M = 2718, N = 304, K = 3024 14.8 | 11.5; M =
// 3628, N = 432, K = 5360 26.1 | 17.6; 181 drawn shapes: 0.88 of the time, the fastest of all kernels on 163, 13 % behind at most;
// up to 576 channels at K < 1600 2 to 5 % behind 64 x 64 ones, M = 2469, N = 448, K = 1280 7.1 | 7.4; behind below, M = 1135,
// N = 1024, K = 1216 7.2 | 7.4, and where a round of 64 x 64 tiles holds the product, M = 182, N = 4480, K = 1984 7.6 | 9.1).
bool oblong_ring_first(int64_t M, int64_t N, int64_t K, int64_t ldx) {
  return K >= 1280 && ceil_div(M, 64) * ceil_div(N, 64) > 256 && oblong_ring(M, N, K, ldx, 64, 128);
}
double rounds_time(const TileRate& r, int64_t M, int64_t N, int64_t K) {
  const double st = static_cast<double>(ceil_div(K, kBK)), round = 256.0 * r.on_cu;
  const int64_t tiles = ceil_div(M, r.bm) * ceil_div(N, r.bn);
  const int64_t full = (tiles - 1) / static_cast<int64_t>(round);
  const double u = (static_cast<double>(tiles) - static_cast<double>(full) * round) / 256.0;
  return r.start + r.per_u * u + static_cast<double>(full) * (r.fill + r.full * st) + st * std::max(r.floor, r.rate0 + r.rate1 * u);
}
// Beyond K = 2560 only one round of 64 x 64 tiles (weights from memory: M = 783, N = 1856, K = 3584, 377 tiles, 18.8
// against 19.9 us), and no few rows (two wave groups are ahead: M = 57, N = 10915, K = 2816 9.8 against 11.6).
bool rounds_modelled(int64_t M, int64_t N, int64_t K) {
  if (N > 16384) return false;  // (beyond what was fitted)
  return K <= 2560 || (K <= kRoundsMaxK && M > 64 && ceil_div(M, 64) * ceil_div(N, 64) <= 256);
}
// cfg: what the thresholds chose.  It stays where it is one of the modelled tiles and less than 5 % behind (the kernels with
// all of K in LDS up to K = 256 are ahead: M = 1502, N = 768, K = 256 3.9 against 4.1 us).
int tile_by_rounds(int cfg, bool onepass, int64_t M, int64_t N, int64_t K) {
  const bool tile = cfg == 1 || cfg == 2 || cfg == 3 || cfg == 6 || cfg == 7 || cfg == 14 || cfg == 17 || cfg == 19 ||
                    cfg == 22 || cfg == 27 || (cfg == 23 && (!onepass || K > 256)) || (cfg == 21 && K > 256 && K <= kOnePassMaxK);
  if (!tile || !rounds_modelled(M, N, K)) return cfg;
  int best = cfg;
  double least = 1e30;
  const auto offer = [&](const TileRate& r) {
    const double us = rounds_time(r, M, N, K) * (r.cfg == cfg || (r.cfg == 17 && cfg == 19) ? 0.95 : 1.0);
    if (us < least) {
      least = us;
      best = r.cfg;
    }
  };
  if (K <= 2 * kBK)
    for (const TileRate& r : kShortRates) offer(r);
  else
    for (const TileRate& r : kRates) offer(r);
  // (one round of 128 x 256: copies two stages wide from K = 1104 on, us, one stage | two: M = 2224, N = 3040, K = 1400
  // 17.9 | 16.5, M = 2032, N = 2704, K = 1720 16.7 | 15.9, M = 517, N = 7344, K = 1056 level, M = 353, N = 12032, K = 832 11.6 |
  // 11.0, M = 669, N = 7296, K = 896 10.2 | 10.8)
  return best == 17 && (cfg == 19 || (K >= 1104 && ceil_div(M, 128) * ceil_div(N, 256) <= 256)) ? 19 : best;
}

// One round of 64 x 64 tiles beyond the shapes that tile_by_rounds models: the lone tile's ring of six stages is ahead of two
// wave groups (cfg 2, 14) and of the kernel whose waves take their weights through registers (27), which wait for their
// stages in registers or for the weights they asked for at once (us, weights from memory, those | the ring: 1452 x 4016 -> 369
// 14.1 | 11.3, 759 x 4432 -> 960 13.6 | 11.6, 173 x 7264 -> 4026 22.9 | 20.3, 1418 x 7088 -> 512 19.4 | 16.5, 49 x 3408 -> 8256 15.3 |
// 13.0, 88 x 4352 -> 8192 level at 14.0; 70 shapes drawn over K = 1100 ... 14000: never more than 3 % behind, 6 % ahead on average).
bool lone_ring_first(int cfg, const LinearQuery& q) {
  return (cfg == 2 || cfg == 14 || cfg == 27) && one_round_ring(q.M, q.N, q.K) && dma_limits_ok(q.K, q.ldx);
}

// forced: tmq_linear_desc::kernel - 1 (-1 = automatic choice).
LinearChoice choose_linear(const LinearQuery& q, int forced) {
  LinearChoice c;
  if (!q.vec_ok || forced == 9) {
    c.cfg = 9;
    return c;
  }
  if (forced < 0 && huge_n_tiles_preferred(q)) {
    c.cfg = 23;
    return c;
  }
  if (forced < 0 && resident_preferred(q)) {
    c.cfg = 28;
    return c;
  }
  if (forced < 0 && onepass_limits_ok(q) && wloop_tile(q.M, q.N, q.K) != 0) {
    c.cfg = wloop_tile(q.M, q.N, q.K) == 32 ? 29 : 30;
    return c;
  }
  const bool stream_auto =
      forced < 0 && (q.M <= kDecodeRowsAuto ||
                     (q.M <= kDecodeMaxRows &&
                      small_rows_path(q.M, q.N, q.K, q.workspace_attached && q.K % 16 == 0) == SmallRows::kStream));
  if (stream_auto || forced == 8) {
    c.cfg = stream_limits_ok(q) ? 8 : kNoKernel;
    return c;
  }
  const bool dma_ok = dma_limits_ok(q.K, q.ldx);
  if (forced < 0 || forced == 13) {
    const SplitPlan p = forced == 13 ? plan_split_tiles(q.M, q.N, q.K) : plan_split(q.M, q.N, q.K);
    if (p.splits > 1 && q.workspace_bytes >= split_workspace_bytes(p, q.M) &&
        (forced == 13 || q.mode == kOutAcc32 || !dma_ok || !ring_ahead_of_split(q.M, q.N, q.K))) {
      c.cfg = 13;
      c.split = p;
      return c;
    }
    if (forced == 13) return c;
  }
  const bool onepass_ok = onepass_limits_ok(q);
  const int64_t M = q.M, N = q.N, K = q.K;
  int cfg = forced;
  if (cfg < 0 && onepass_ok && K <= kOnePassMaxK && ceil_div(M, 64) * ceil_div(N, 64) <= 256) {
    // short K on a grid no larger than the chip: one latency instead of one per stage
    // (M = 128, K = N = 1024: 6.0 -> 5.6 us with cold weights); up to 512 tiles of 32 x 32
    // whose waves split K spread the copies over more CUs (3.8 us; M = 512: 5.7 -> 4.4 us;
    // N = 4096, K = 512, M = 128: 4.4 -> 4.3 us; 640 tiles and more: tile_by_rounds; K <= 256: slower)
    cfg = K > 256 && ceil_div(M, 32) * ceil_div(N, 32) <= 512 ? 24 : 21;
  } else if (cfg < 0 && onepass_ok && onepass_wide_preferred(M, N, K)) {
    cfg = 23;
    c.onepass = true;
  } else if (cfg < 0 && onepass_ok && wstream_tile(M, N, K) != 0) {
    // K up to 4096 on a grid of 32 x 32 tiles that the chip holds at once: the waves split
    // K and take their weights through registers (cold weights, K = N = 4096, M = 64:
    // 12.2 -> 8.6 us; K = 2048, N = 4096: M = 64 9.4 -> 5.5 us, M = 128 9.4 -> 7.0 us;
    // K = N = 2048: M = 128 7.8 -> 5.0 us, M = 256 8.0 -> 6.3 us)
    cfg = wstream_tile(M, N, K) == 32 ? 25 : 26;
  } else if (cfg < 0) {
    // Thresholds from timing sweeps over M, N, K on the chip (256 CUs, cold weights): the
    // 256x256 tile (one block per CU) wins from 129 tiles on, the 128x256 tile while
    // it fits one round, the 128x128 tile (two blocks per CU) down to 128 tiles.
    const auto nblk = [&](int bm, int bn) { return ceil_div(M, bm) * ceil_div(N, bn); };
    // (and only when the rows fill at least 55 % of the row tiles: a tile's time
    // does not shrink with its padding; M = 100 and 150 against N = 49152 sit on
    // either side)
    const auto rows_used = [&](int bm) { return M * 20 >= ceil_div(M, bm) * bm * 11; };
    // One block of either large tile runs per CU.  The 128x256 tile (128 activation rows,
    // 256 channels; 8 waves of 64x64) keeps a single round to itself (M = 2048, N = 4096,
    // 256 tiles: 34.4 us against 40.1 us for 128 tiles of 256x256); once it needs a second
    // round the 256x256 tiles take over (M = 768, N = 11008, 129 tiles: 43.4 against 49.4 us;
    // M = 3072, K = N = 3072, 144 tiles: 34.3 against 39.1 us), except just past a full round
    // of them, where the second round of 256x256 tiles is nearly empty and three rounds of
    // 128x256 are shorter (258 tiles, M = 1536, N = 11008: 84.9 against 91.8 us; 344 tiles:
    // 90.6 against 91.6 us; at 375 ... 384 tiles the two are within 4 % of each other, either
    // way round from box to box; 430 tiles: 102.4 against 115.8 us; at 516 tiles, just past
    // two rounds, the two are level: 146.8 against 146.3 us).  Its
    // mirror image, 256 rows x 128 channels, is 17 % slower than 256x256 at C3: activation
    // rows arrive as 64-byte pieces of far-apart rows, weight rows as 256-byte pieces of
    // the packed layout.
    const int64_t t256 = nblk(256, 256), t128x256 = nblk(128, 256);
    // (the 128x256 tile's activation copies two stages wide pay within one round of tiles only:
    // M = 512, N = 11008: 36.3 -> 32.7 us, but M = 1024, N = 11008: 53.0 -> 57.7 us)
    const int cfg128x256 = t128x256 <= 256 ? 19 : 17;
    // equal tile counts: the 64 x 128 tile; more row tiles than its mirror image has fewer
    // blocks and idle CUs (M = 192: N = 6144, K = 3072: 17.1 against 15.3 us with 128 x 64;
    // N = 4096, K = 11008: 46.8 against 43.4 us); up to 96 rows fill three of the 128 x 64 tile's
    // four row strips and it is ahead at equal counts too (M = 96, N = 13824, K = 5120: 28.4
    // against 31.0 us; N = 11008, K = 4096: 20.2 against 21.2 us)
    const int cfg_half =
        nblk(128, 64) <= 256 && (nblk(128, 64) > nblk(64, 128) || (M <= 96 && nblk(128, 64) == nblk(64, 128))) ? 22 : 23;
    // Just past a round of 128 x 128 tiles, half a round of 128 x 256 ones is ahead behind many rows (us, 128 x 128 | 128 x 256:
    // M = 2798, N = 1536, K = 4160 0.80 of the time, M = 3613, N = 1216, K = 4288 33.5 | 26.3; M = 2613, N = 1792, K = 6800 0.87, M =
    // 3379, N = 1344, K = 7760 0.73), up to 2560 of them while K is no longer than 6144 (M = 1779, N = 2544, K = 7424 49.3 | 51.8,
    // M = 2018, N = 2432, K = 7616 1.04 times, M = 1732, N = 2768, K = 7168 48.2 | 49.6).
    const bool rows_ahead = M >= 1536 && K <= (M < 2560 ? 6144 : 8192);
    // Many rows against a short K are bound by the epilogue, and 256-channel tiles requantise the padding behind
    // N as well: 128 x 128 tiles where those pad a quarter less (M = 100352 pixels of a 56 x 56 feature map at batch
    // 32: N = 384, K = 96: 35.1 -> 27 us; N = 96, K = 384: 20.9 -> 15.7 us; N = 512, K = 128 has nothing to gain and
    // stays: 10.4 against 12.5 us).
    const bool padding_bound = K <= 512 && round_up(N, 256) * 4 >= round_up(N, 128) * 5;
    if (t128x256 > 256 && rows_used(256) && padding_bound)
      cfg = 7;
    else if (t128x256 > 256 && rows_used(256))
      cfg = t256 > 256 && t256 <= 400 ? 17 : 6;  // 6: 8 waves of 128x64, operands copied straight into LDS
    else if (t128x256 >= 160 && rows_used(128))
      // (barely more than half a round of them, against a long K and not too many rows: 128x128 tiles, at most 320 (304),
      // all resident at once; the branch of 128x128 tiles below has the figures)
      cfg = K >= 4096 && nblk(128, 128) <= (M < 576 ? 304 : 320) && !rows_ahead ? 7 : cfg128x256;
    else if (N >= 2048 && (N >= 4096 || K >= 4096) && nblk(64, 64) > 256 && (nblk(64, 128) <= 256 || M <= 64))
      // a few hundred rows whose 128 x 128 tiles would leave half the chip idle and whose
      // 64 x 64 tiles need a second round: 64 rows x 128 channels, one round (K = N = 4096,
      // cold weights: M = 448: 24.6 -> 19.1 us, M = 512: 24.8 -> 19.3 us; K = 2048: 14.7 -> 11.7 us;
      // N = 8192, M = 192: 25.9 -> 19.9 us; against N = 1024 the 128 x 128 tiles stay ahead:
      // M = 1536, K = 4096: 17.4 against 20.2 us, and at K = N = 2048, M = 1024: 11.5 against 12.2 us);
      // up to 64 rows also over several rounds, ahead of 128 x 128 tiles that are three quarters padding
      // (M = 32, K = 4096: N = 65536 48.2 against 53.4 us, N = 128256 87.7 against 95 us; K = 2048, N = 65536:
      // 26.5 against 30.8 us; N = 49152: level)
      cfg = cfg_half;
    else if (N >= 2048 && (N >= 4096 || K >= 4096) && nblk(64, 64) > 256 && nblk(128, 64) <= 256)
      cfg = 22;
    else if (nblk(128, 128) >= 128 && M > 64)  // (64 tiles: 64x64 wins, 15.2 against 17.9 us at M = 256, K = N = 4096;
                                               // up to 64 rows half of every tile is padding: M = 64, N = 16384, K = 4096:
                                               // 27.5 us against 17.5 us for the 64 x 64 tiles that walk K in phases)
      // (just past a round of them 128 x 256 ones are more than half a round.  Up to 320 tiles (304 below 576 rows), us, 128 x 128 |
      // 128 x 256: M = 374, N = 12208, K = 8304 65 | 76, M = 887, N = 5280, K = 3520 28.7 | 30.3, M = 1234, N = 3440, K = 4992 33.8 | 36.5,
      // M = 640, N = 8192, K = 4096 29.3 | 31.3, M = 1650, N = 2512, K = 8960 55.2 | 61.3; on 118 drawn shapes of that kind 128 x 128
      // are 1 % ahead on average, 12 % at most, and up to 44 % behind with 1040 to 1536 rows at K below 4000 (M = 1209, N = 3328,
      // K = 3520 28.1 | 22.9, M = 1168, N = 3728, K = 2640 24.7 | 22.0) or more than 2688 past K = 8192 (M = 2722, N = 1456, K =
      // 9232 73 | 51), which no line here tells apart yet.  The other side of the lines: 11 % ahead on 176, 6 % behind at most;
      // M = 479, N = 9984, K = 2816 27.8 | 24.9, M = 490, N = 10032, K = 5440
      // 50.1 | 46.0, M = 695, N = 8688, K = 5824 53.1 | 47.2, M = 2547, N = 1680, K = 4592 39.0 | 27.9)
      cfg = K > 2560 && nblk(128, 128) > 256 && rows_used(128) && (nblk(128, 128) > (M < 576 ? 304 : 320) || rows_ahead) ? cfg128x256 : 7;
    else if (onepass_ok && K >= 3072 && K <= kWringMaxK && nblk(64, 64) <= 256 && N * K <= (int64_t{3} << 23))
      // one round of 64 x 64 tiles against a long K: eight waves split K, weights through
      // registers, activations through a ring per wave, no barrier before the partial tiles
      // meet (cold weights, K = N = 4096: M = 130 12.1 -> 11.8 us, M = 192 14.0 -> 12.8 us,
      // M = 256 14.3 -> 13.6 us; N = 2048: M = 512 14.0 -> 13.0 us; K = 3072: M = 192
      // 13.0 -> 12.1 us; behind the two wave groups at K = 2560 (12.3 against 11.7 us) and
      // against 32 MB of weights, N = 8192: 15.3 against 14.6 us; 24 MB, N = 6144, K = 4096,
      // M = 128: 13.7 against 15.0 us).  Raw accumulators; lone_ring_first takes bytes and floats
      cfg = 27;
    else if (onepass_ok && phased_ring_preferred(M, N, K))
      cfg = 21;
    else if (nblk(64, 64) <= 256 && ceil_div(K, kBK) >= 32 && ceil_div(K, kBK) % 2 == 0)
      cfg = 14;  // at most one block per CU and a long k loop: two wave groups halve it (14.7 -> 11.7 us
                 // at M = 128, K = N = 4096; four groups run into the L2's bandwidth: 12.3 us); raw
                 // accumulators here and below, lone_ring_first takes bytes and floats
    else {
      cfg = 2;
      c.groups = two_wave_groups_fit(M, N, K) ? 2 : 1;  // (an odd number of stages, or a shorter loop)
    }
  }
  if (forced < 0 && q.mode != kOutAcc32 && dma_limits_ok(std::max<int64_t>(K, 3 * kBK), q.ldx)) {
    const int by_rounds = tile_by_rounds(cfg, c.onepass, M, N, K);
    if (by_rounds != cfg) c.onepass = false;
    if (by_rounds == 2 && rounds_modelled(M, N, K)) c.groups = 1;
    cfg = by_rounds;
  }
  if (forced < 0 && q.mode != kOutAcc32 && lone_ring_first(cfg, q)) {
    cfg = 2;
    c.groups = 1;
  }
  if (forced < 0 && q.mode != kOutAcc32 && (cfg == 1 || cfg == 2 || cfg == 7 || cfg == 14 || cfg == 17) &&
      oblong_ring_first(M, N, K, q.ldx)) {
    cfg = 23;
    c.groups = 1;
  }
  const bool wide_ok = wide_limits_ok(K, q.ldx);
  if (cfg == 19 && !wide_ok) cfg = 17;
  // 256 x 256 tiles with byte or float outputs: the persistent kernel, which hides each
  // tile's pipeline fill behind the tile before it and whose epilogue needs no block
  // barrier (also ahead on a single round: M = N = K = 4096, 256 tiles: 61.9 -> 59.7 us;
  // 2560 x 4096: 46.4 -> 45.8 us; never behind in a sweep of one to three rounds)
  if (forced < 0 && cfg == 6 && wide_ok && q.mode != kOutAcc32) cfg = 20;
  if (cfg == 20 && q.mode == kOutAcc32) cfg = 6;  // raw outputs: one tile per block
  if (cfg == 20 && !wide_ok) cfg = 3;
  if (cfg == 6 && !wide_ok) cfg = 3;
  if (cfg == 17 && !dma_ok) cfg = 3;
  if (cfg == 7 && !wide_ok) cfg = 1;
  switch (cfg) {
    case 0: case 1: case 2: case 3: case 4: case 5: case 6: case 7: case 17: case 19: case 20: case 22: case 23:
      break;
    case 14:  // two wave groups: equal runs of stages only
      if (ceil_div(K, kBK) % 2 != 0) cfg = kNoKernel;
      break;
    case 21:
      if (!onepass_ok) cfg = kNoKernel;
      break;
    case 24:
      if (!onepass_ok || K > kOnePassMaxK) cfg = kNoKernel;
      break;
    case 25: case 26:
      if (!onepass_ok || K > 4096) cfg = kNoKernel;
      break;
    case 27:
      if (!onepass_ok || K > kWringMaxK) cfg = kNoKernel;
      break;
    case 28:
      if (!resident_limits_ok(M, N, K, q.ldx, 256)) cfg = kNoKernel;
      break;
    case 29: case 30:
      if (!onepass_ok) cfg = kNoKernel;
      break;
    default:
      cfg = kNoKernel;
  }
  c.cfg = cfg;
  return c;
}

// More than 16 rows off the 16-byte grid, one round of tiles of 32 rows: eight waves a tile that walk K in pieces and read the rows
// where they lie (gemm_i8_wloop.h has both sides).  Tiles of 64 channels, whose pieces are half as long, where not every wave would
// have one otherwise (us, 32 | 64 channels: 24 x 276 -> 65 3.8 | 3.6, 1279 x 378 -> 64 4.0 | 3.8; 523 x 360 -> 322 level; 205 x 684
// -> 640 4.0 | 4.1) and where 32 do not fit a round.  Two stages and less stay with the 64 x 64 tiles (those | these: 172 x 84 -> 64
// 3.3 | 3.6, 1897 x 76 -> 128 3.5 | 3.7, 136 x 88 -> 1043 3.7 | 3.9; 97 x 152 -> 64 3.6 | 3.4, 26 x 132 -> 8064 4.1 | 3.7).  Returns the
// channels per tile, 0: not such a shape.
constexpr int64_t kWloopRaggedMinK = 2 * kBK, kWloopRaggedShortK = 512;
int wloop_ragged_tile(int64_t M, int64_t N, int64_t K) {
  if (M <= kDecodeRowsAuto || K <= kWloopRaggedMinK || K > kWloopMaxK || ceil_div(M, 32) * ceil_div(N, 64) > 256) return 0;
  return K > kWloopRaggedShortK && ceil_div(M, 32) * ceil_div(N, 32) <= 256 ? 32 : 64;
}

// ... but for rows that the streaming kernel takes on the grid: a copy in front of that is ahead, if there is room for it, where rows
// off the 4-byte grid, whose requests cost twice as much, are long and the weights many (an operator's call after the other, us, in
// place | copied: 24 x 8001 -> 2600 15.7 | 13.0, 17 x 6001 -> 2600 11.1 | 9.8, 24 x 11001 -> 1000 18.0 | 14.4, 24 x 12001 -> 4000 22.1 |
// 18.9, 28 x 10001 -> 2600 18.5 | 16.7; at odd lengths up to 8192 of few weights as well, 24 x 8001 -> 64 12.8 | 11.2, 22 x 7929 -> 37 12.6 |
// 10.4, 20 x 7001 -> 300 11.6 | 10.4, 17 x 8001 -> 17 10.4 | 10.2).  The other side: 28 x 7001 -> 1000 11.6 | 12.1; on the device 24 x 5001 ->
// 2600 11.1 | 11.4, 32 x 10001 -> 2600 19.0 | 18.5, 32 x 8001 -> 64 12.8 | 13.9, 24 x 9001 -> 1000 14.2 | 15.1, 24 x 10002 -> 300 13.9 |
// 14.6, and rows on the 4-byte grid, 20 x 5784 -> 51 7.7 | 10.0, 25 x 10116 -> 287 10.7 | 15.4, 22 x 10156 -> 2618 15.4 | 16.5.
constexpr int64_t kFewRowsCopied = 28, kFewRowsCopiedMinK = 5632, kFewerRowsCopied = 24, kFewerRowsCopiedMaxK = 8192;
bool few_rows_copied(int64_t M, int64_t N, int64_t K) {
  return M > kDecodeRowsAuto && M <= kFewRowsCopied && K > kFewRowsCopiedMinK && K % 4 != 0 &&
         (N * K > int64_t{10} << 20 || (K % 2 != 0 && K <= kFewerRowsCopiedMaxK && M <= kFewerRowsCopied)) &&
         small_rows_path(M, N, regrid_pitch(K), true) == SmallRows::kStream;
}
// Whether a copy, if there is room for it, comes before the tiles that wloop_ragged_tile names.
bool wloop_ragged_copied(int64_t M, int64_t N, int64_t K) { return wloop_tile(M, N, regrid_pitch(K)) != 0 || few_rows_copied(M, N, K); }

// More than that: tiles that read the rows where they lie, or a copy onto the grid and the padded shape's own kernel.  The copy is a
// launch (2.2 us and a scratch allocation).
//
// 64 x 64 tiles request every row once per 64 channels, and what bounds them is those unaligned requests; larger tiles halve them and
// cost idle CUs where their grid is short.  So each tile is taken while its own grid makes one round and the smaller one's does not (us,
// the route before (64 x 64, from 512 of them on the copy, K <= 768: 1024) | this one; 200 shapes drawn over M = 100 ... 4096, K = 141 ...
// 4000, N = 240 ... 12000, 65 ... 4200 tiles of 64 x 64; bytes where nothing else is said, floats the same but for the lines that name them):
//   64 x 128 from K = 1200 on (floats 1536: 183 x 1288 -> 6551 9.3 | 10.1, 183 x 1791 -> 5724 11.8 | 11.6): 2106 x 2839 -> 539 19.1 |
//     14.1, 746 x 2053 -> 2555 13.7 | 11.9, 212 x 1481 -> 6574 11.5 | 10.2, 168 x 3495 -> 8678 level at 15.8; below, 64 x 64 are level
//     or up to 12 % ahead (517 x 1000 -> 2051 7.8 | 8.0, 456 x 200 -> 3197 4.9 | 5.5);
//   128 x 128, eight waves: 3931 x 2345 -> 881 24.7 | 16.9, 3819 x 1352 -> 998 19.1 | 12.3, 1989 x 375 -> 1580 9.3 | 7.2, 1019 x 1685 -> 2890
//     15.3 | 13.8, 823 x 3208 -> 3743 21.6 | 19.7; beyond K = 3300 the copy, which floats want (275 x 3317 -> 7349 20.4 | 22.4),
//     up to 256 rows beyond K = 2000 (210 x 2773 -> 11089 17.3 | 18.4, 221 x 2102 -> 8984 14.0 | 14.7); up to 288
//     tiles of 64 x 128 at K <= 640 64 x 64 (230 x 264 -> 9105 5.7 | 6.0), up to 370 at K <= 330 and of floats (837 x 312 -> 2930
//     5.8 | 6.2, bf16 2764 x 417 -> 949 8.7 | 9.2; 1550 x 279 -> 2151, 425 of them, 7.6 | 6.7);
//   128 x 256, eight waves: 1860 x 574 -> 3469 17.8 | 11.8, 4022 x 1928 -> 1556 28.2 | 21.7, 446 x 1309 -> 10760
//     16.8 | 15.8; up to 700 tiles of 64 x 128 at K < 480 those (516 x 372 -> 7244 10.7 | 8.0, with 128 x 256 9.4); up to 512 rows beyond
//     K = 2000 the copy, whose time follows the rows (copied | 128 x 256: 264 x 2227 -> 12681 23.7 | 25.6, 399 x 2179 -> 12067 24.5 | 26.2,
//     471 x 3206 -> 8959 32.3 | 36.0, 500 x 2302 -> 11735 26.4 | 28.9, 499 x 2209 -> 11550 level, 494 x 3272 -> 15876 38.8 | 39.2; the other
//     side 449 x 1113 -> 11446 18.2 | 17.0, 566 x 2942 -> 10913 34.0 | 32.5, 654 x 3138 -> 6707 31.4 | 32.5);
//   beyond one round of those 128 x 128 where the copy is not ahead, K = 250 ... 640 (1356 x 344 -> 7817 17.3 | 14.4, 3508 x 252 -> 4716
//     20.4 | 17.2; 1258 x 333 -> 9024 12.9 | 13.4; 7202 x 245 -> 1879 15.9 | 16.7, 2759 x 2023 -> 3364 34.9 | 38.1), of bytes beyond
//     K = 400 only up to 200 tiles of 256 x 256, which on the grid fill a round from there on (their tiles: 216, 2034 x 637 -> 6687 22.1 |
//     25.8; 216, 897 x 577 -> 13709 20.8 | 23.3; 220, 2546 x 635 -> 5628 22.4 | 25.1; 240, 3014 x 405 -> 4927 19.1 | 20.6; 245, 1655 x 537 ->
//     8955 22.5 | 25.3; 280, 1037 x 421 -> 14325 18.7 | 21.7; the mean of 26 drawn ones 1.05; the other side: 204, 1356 x 561 -> 8586 21.0 |
//     19.5; 215, 1151 x 504 -> 10801 19.6 | 17.4; 152, 965 x 332 -> 9627 17.7 | 14.6; 168, 1963 x 522 -> 5352 20.4 | 17.6; floats 0.59 to 0.89
//     but for 3293 x 324 -> 2880 1.06).
// Elsewhere 64 x 64 up to 512 tiles, later where K is short, beyond that the copy (direct | copy: K = 2051, N = 1000, M = 517 9.3 |
// 10.7; K = 4100, N = 3900, M = 500 22.6 | 23.9; K = 3907, N = 193, M = 2889 13.6 | 25.3; K = 100, N = 1000, M = 8000 10.4 | 12.8; K = 120,
// N = 8000, M = 4096 26.3 | 22.1).
enum class RaggedTile { kCopy, k64, k64x128, k128, k128x256 };
constexpr int64_t kRaggedLargeMaxTiles = 4096, kRaggedLargeMaxK = 4000, kRagged128MaxK = 3300, kRagged128FewRowsMaxK = 2000;
// room: for the copy; without it the larger tiles take the last two kinds of shapes as well.
RaggedTile ragged_tile(int64_t M, int64_t N, int64_t K, bool floats, bool room) {
  if (K < 16 || K > 0x7fffff00) return RaggedTile::kCopy;
  if (M <= kDecodeMaxRows && small_rows_path(M, N, regrid_pitch(K), true) == SmallRows::kStream) return RaggedTile::kCopy;
  const int64_t rows64 = ceil_div(M, 64), rows128 = ceil_div(M, 128);
  const int64_t tiles = rows64 * ceil_div(N, 64), oblong = rows64 * ceil_div(N, 128);
  const bool one128 = rows128 * ceil_div(N, 128) <= 256;
  // (at least 96 rows and 384 channels: fewer are padding in the larger tiles, 9974 x 296 -> 289 8.1 | 8.5)
  if (tiles > 256 && tiles <= kRaggedLargeMaxTiles && M >= 96 && N >= 384 && K > 2 * kBK &&
      K <= (oblong <= 256 ? kRaggedLargeMaxK : M > (one128 || !room ? 256 : 512) ? kRagged128MaxK : kRagged128FewRowsMaxK)) {
    if (oblong <= 256) {
      if (K > (floats ? 1536 : 1200)) return RaggedTile::k64x128;
    } else if (one128) {
      if (K > 640 || oblong > (K > 330 && !floats ? 288 : 370)) return RaggedTile::k128;
    } else if (rows128 * ceil_div(N, 256) <= 256) {
      return K >= 480 || oblong > 700 ? RaggedTile::k128x256 : RaggedTile::k64x128;
    } else if (K >= 250 && K <= 640 && (floats || !room || K <= 400 || ceil_div(M, 256) * ceil_div(N, 256) <= 200)) {
      return RaggedTile::k128;
    }
  }
  return tiles <= (K <= 128 ? 3072 : K <= 768 ? 1024 : 512) ? RaggedTile::k64 : RaggedTile::kCopy;
}

// ... and where the copy comes before 64 x 64 tiles, if there is room for it: K so long that the padded shape's kernel earns it back (two
// layers, quantize and dequantize as a program calls them, direct | copy, us; 64 x 128 tiles in a ring: 600 x 6001 -> 2000
// 45.3 | 34.6).  One round of tiles of 32 rows against K > 4096 reads the rows in place where there is no room (wloop_ragged_tile),
// which operators leave out there: a caller that gives the room tmq_linear_scratch_bytes names has them copied.  Copied over in place on
// the device, 188 drawn shapes of more than 32 rows: even K 1.06 to 1.13 of the time by range of K, odd K 1.06 to 1.10 up to 6000, level up to
// 8000, 0.93 to 0.97 beyond (0.81 to 1.28 there); the copy's launch and memory are the host's besides.
bool ragged_copy_first(int64_t M, int64_t N, int64_t K) {
  const int64_t pitch = regrid_pitch(K);
  return wloop_tile(M, N, pitch) != 0 || (K >= 2304 && oblong_ring_first(M, N, pitch, pitch));
}
RaggedTile ragged_route(int64_t M, int64_t N, int64_t K, bool floats, bool copy_ok) {
  const RaggedTile tile = ragged_tile(M, N, K, floats, copy_ok);
  return tile == RaggedTile::k64 && copy_ok && ragged_copy_first(M, N, K) ? RaggedTile::kCopy : tile;
}

template <int MODE>
int dispatch_linear(const GemmArgs& a, const XLinear& xs, int x_signed, bool vec_ok, int forced,
                    hipStream_t s, void* workspace = nullptr, int64_t workspace_bytes = 0) {
  LinearQuery q;
  q.M = a.M;
  q.N = a.N;
  q.K = a.K;
  q.ldx = xs.ldx;
  q.n_off = a.n_off;
  q.mode = MODE;
  q.vec_ok = vec_ok;
  q.workspace_attached = workspace != nullptr;
  q.workspace_bytes = workspace != nullptr && aligned(workspace, 16) ? workspace_bytes : 0;
  if (a.splits != 1) return TMQ_ERR_INVALID_ARGUMENT;  // the split is this function's to plan
  if (!vec_ok && forced < 0) {
    // Off the 16-byte grid: up to 16 rows stream the weights as they are (the copy would cost a
    // launch, more than any other kernel's advantage at so few rows); more rows take tiles
    // that read them where they lie, or are copied onto the grid if the caller left room for that
    // and take the kernel of the padded shape.
    if (a.M <= kDecodeRowsAuto && a.K >= 16 && stream_limits_ok(q) && a.w_kchunks == packed_kchunks(a.K))
      return launch_linear_decode_ragged<MODE>(a, xs, s);
    const int64_t room = regrid_bytes(a.M, a.K);
    const bool copy_ok = regrid_limits_ok(a.M, a.K) && q.workspace_bytes >= room;
    const bool zero_padded = a.w_kchunks == packed_kchunks(a.K);
    if (const int tile = wloop_ragged_tile(a.M, a.N, a.K); tile != 0 && zero_padded && xs.ldx <= (int64_t{1} << 23) &&
        a.N + a.n_off < (int64_t{1} << 29) && !(copy_ok && wloop_ragged_copied(a.M, a.N, a.K)))
      return launch_gemm_wloop_ragged<MODE>(a, xs, tile == 64, s);
    const XLinearRagged rows{xs.x, xs.ldx};
    switch (zero_padded ? ragged_route(a.M, a.N, a.K, MODE == kOutF32, copy_ok) : RaggedTile::kCopy) {
      case RaggedTile::k64:
        return two_wave_groups_fit(a.M, a.N, a.K) ? launch_gemm<64, 64, 2, 2, MODE, 4, false, 2>(a, rows, s)
                                                  : launch_gemm<64, 64, 2, 2, MODE>(a, rows, s);
      case RaggedTile::k64x128: return launch_gemm<64, 128, 2, 2, MODE>(a, rows, s);
      case RaggedTile::k128: return launch_gemm<128, 128, 2, 4, MODE>(a, rows, s);
      case RaggedTile::k128x256: return launch_gemm<128, 256, 2, 4, MODE>(a, rows, s);
      case RaggedTile::kCopy: break;
    }
    if (copy_ok) {
      const int rc = launch_regrid(xs, a.M, a.K, workspace, s);
      if (rc != TMQ_OK) return rc;
      GemmArgs b = a;
      b.K = regrid_pitch(a.K);  // (the packed weights are zero from K on, up to a multiple of 128)
      const XLinear on_grid{static_cast<const uint8_t*>(workspace), b.K};
      const bool rest = workspace_bytes > room;
      return dispatch_linear<MODE>(b, on_grid, x_signed, true, forced, s,
                                   rest ? static_cast<uint8_t*>(workspace) + room : nullptr,
                                   rest ? workspace_bytes - room : 0);
    }
  }
  const LinearChoice c = choose_linear(q, forced);
  switch (c.cfg) {
    case 9: {
      // plain kernel accumulates true activation values: undo the +128 share
      GemmArgs b = a;
      if (!x_signed) {
        b.acc_coef -= 128;
        b.acc_base -= 128;
      }
      const int64_t work = a.M * ceil_div(a.N, 4);
      const int64_t blocks = ceil_div(work, 256);
      if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
      enqueue(linear_plain_kernel<MODE>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, b, xs, x_signed);
      return launch_status();
    }
    case 8: return launch_linear_decode<MODE>(a, xs, s);
    case 28: {
      const int rc = launch_linear_resident<MODE>(a, xs, s);
      // (a device with too few CUs for this many channel groups: the automatic choice streams instead)
      return rc == TMQ_ERR_UNSUPPORTED && forced < 0 && stream_limits_ok(q) ? launch_linear_decode<MODE>(a, xs, s) : rc;
    }
    case 13: return run_split<MODE>(a, xs, c.split, workspace, dma_limits_ok(a.K, xs.ldx), s);
    case 0: return launch_gemm<256, 256, 2, 2, MODE>(a, xs, s);
    case 1: return dma_limits_ok(a.K, xs.ldx) ? launch_gemm_any_size<128, 128, 2, 2, MODE, 3, true>(a, xs, s)
                                              : launch_gemm_any_size<128, 128, 2, 2, MODE>(a, xs, s);
    case 2: return c.groups == 2                  ? launch_gemm<64, 64, 2, 2, MODE, 4, false, 2>(a, xs, s)
                   : one_round_ring(a.M, a.N, a.K) && dma_limits_ok(a.K, xs.ldx)
                       ? launch_gemm<64, 64, 2, 2, MODE, 6, true>(a, xs, s)
                   : dma_limits_ok(a.K, xs.ldx) ? launch_gemm_any_size<64, 64, 2, 2, MODE, 3, true>(a, xs, s)
                                                : launch_gemm_any_size<64, 64, 2, 2, MODE>(a, xs, s);
    case 3: return launch_gemm_any_size<256, 256, 2, 4, MODE, 3>(a, xs, s);
    case 4: return launch_gemm<128, 256, 2, 2, MODE>(a, xs, s);
    case 5: return launch_gemm<256, 128, 2, 2, MODE>(a, xs, s);
    case 6: return launch_gemm<256, 256, 2, 4, MODE, 3, true, 1, true>(a, xs, s);
    // (a block per CU: eight waves, so that one's fragment reads run beside another's products, and from K = 1536 on a ring
    // of six stages where the copies of 64 activation bytes lie in one line each.  Us, four waves | eight | eight and six
    // stages: M = 1160, N = 2048, K = 11008 59.4 | 58 | 41.7; M = 1062, N = 2496, K = 6016 35.5 | - | 26.8; M = 617, N = 5952,
    // K = 1728 14.2 | 13.7 | 13.0; M = 752, N = 4800, K = 960 8.7 | 8.0 | 8.4; M = 254, N = 11264, K = 2480 20.3 | 19.8 | 23.5)
    case 7: return ceil_div(a.M, 128) * ceil_div(a.N, 128) > 256
                       ? launch_gemm_any_size<128, 128, 2, 2, MODE, 3, true, true>(a, xs, s)
                   : a.K >= 1536 && a.K % kBK == 0 ? launch_gemm<128, 128, 2, 4, MODE, 6, true>(a, xs, s)
                                                   : launch_gemm<128, 128, 2, 4, MODE, 3, true, 1, true>(a, xs, s);
    case 14: return launch_gemm<64, 64, 2, 2, MODE, 4, false, 2>(a, xs, s);
    case 17: return launch_gemm_any_size<128, 256, 2, 4, MODE, 3, true>(a, xs, s);
    case 19: return launch_gemm<128, 256, 2, 4, MODE, 3, true, 1, true>(a, xs, s);
    case 20: return launch_gemm_persistent<MODE>(a, xs, s);
    case 22: return oblong_ring(a.M, a.N, a.K, xs.ldx, 128, 64) ? launch_gemm<128, 64, 2, 2, MODE, 6, true>(a, xs, s)
                                                                : launch_gemm<128, 64, 2, 2, MODE>(a, xs, s);
    case 23: return c.onepass ? launch_gemm_onepass<MODE, 128>(a, xs, s)
                    : oblong_ring(a.M, a.N, a.K, xs.ldx, 64, 128) ? launch_gemm<64, 128, 2, 2, MODE, 6, true>(a, xs, s)
                                                                  : launch_gemm<64, 128, 2, 2, MODE>(a, xs, s);
    case 21: return launch_gemm_onepass<MODE>(a, xs, s);
    case 24: return launch_gemm_ksplit<MODE>(a, xs, s);
    case 25: return launch_gemm_wloop<MODE>(a, xs, wstream_pairs(a.M, a.N), s);
    case 26: return launch_gemm_wloop<MODE>(a, xs, true, s);
    case 27: return launch_gemm_wring<MODE>(a, xs, s);
    case 29: case 30: return launch_gemm_wloop<MODE>(a, xs, c.cfg == 30, s);
    default: return TMQ_ERR_UNSUPPORTED;
  }
}

int fill_args(const tmq_linear_desc* d, GemmArgs* a, XLinear* xs, bool* vec_ok) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->M < 0 || d->N < 0 || d->K < 0) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->M == 0 || d->N == 0) return TMQ_OK;
  if (d->x == nullptr && d->K > 0) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->w_packed == nullptr || d->w_colsum == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->ldx < d->K) return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(d->w_packed, 16)) return TMQ_ERR_ALIGNMENT;
  a->M = d->M;
  a->N = d->N;
  a->K = d->K;
  a->w_packed = static_cast<const uint8_t*>(d->w_packed);
  a->w_kchunks = packed_kchunks(d->K);
  a->colsum = d->w_colsum;
  a->x_xor = d->x_signed ? 0u : 0x80808080u;
  a->n_off = 0;
  xs->x = static_cast<const uint8_t*>(d->x);
  xs->ldx = d->ldx;
  *vec_ok = d->K >= 16 && d->K % 16 == 0 && d->ldx % 16 == 0 && aligned(d->x, 16);
  return TMQ_OK;
}

}  // namespace
}  // namespace tmq

using namespace tmq;

TMQ_EXPORT int64_t tmq_linear_packed_kchunks(int64_t K) { return K < 0 ? 0 : packed_kchunks(K); }

TMQ_EXPORT int64_t tmq_linear_packed_bytes(int64_t N, int64_t K) {
  if (N < 0 || K < 0) return 0;
  return ceil_div(N, 16) * packed_kchunks(K) * 256;
}

TMQ_EXPORT int tmq_linear_prepack(const int8_t* w, int64_t N, int64_t K, int64_t ldw, void* packed,
                                  int32_t* colsum, tmq_stream_t stream) {
  if (N < 0 || K < 0 || ldw < K) return TMQ_ERR_INVALID_ARGUMENT;
  if (N == 0) return TMQ_OK;
  if (packed == nullptr || colsum == nullptr || (w == nullptr && K > 0))
    return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(packed, 16)) return TMQ_ERR_ALIGNMENT;
  hipStream_t s = as_stream(stream);
  const int64_t KC = packed_kchunks(K);
  const int64_t total = ceil_div(N, 16) * KC * 16;
  const bool vec = aligned(w, 16) && ldw % 16 == 0;
  if (total > 0) {
    const int64_t blocks = ceil_div(total, 256);
    if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
    enqueue(prepack_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s,
            w, N, K, ldw, KC, total, vec, static_cast<uint8_t*>(packed));
    if (launch_status() != TMQ_OK) return TMQ_ERR_LAUNCH;
  }
  const int64_t blocks = ceil_div(N, 256 / kWave);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  enqueue(colsum_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, w, N, K, ldw, vec, colsum);
  return launch_status();
}

TMQ_EXPORT int tmq_linear_unpack(const void* packed, int64_t N, int64_t K, int8_t* w, int64_t ldw,
                                 tmq_stream_t stream) {
  if (N < 0 || K < 0 || ldw < K) return TMQ_ERR_INVALID_ARGUMENT;
  if (N == 0 || K == 0) return TMQ_OK;
  if (packed == nullptr || w == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  const int64_t blocks = ceil_div(N * K, 256);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  enqueue(unpack_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, as_stream(stream),
          static_cast<const uint8_t*>(packed), N, K, ldw, packed_kchunks(K), w);
  return launch_status();
}

TMQ_EXPORT int64_t tmq_linear_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return split_workspace_bytes(plan_split(M, N, K), M);
}

namespace tmq {
namespace {

// Bytes of a split along K that products of bytes or floats on the grid make use of: none where the automatic choice is the
// same kernel with and without them (the plan is there for pinned kernels and raw accumulators).
int64_t split_bytes_used(int64_t M, int64_t N, int64_t K) {
  LinearQuery q;
  q.M = M;
  q.N = N;
  q.K = q.ldx = K;
  q.vec_ok = q.workspace_attached = true;
  q.workspace_bytes = split_workspace_bytes(plan_split(M, N, K), M);
  if (q.workspace_bytes == 0) return 0;
  for (const int mode : {kOutU8, kOutF32}) {
    q.mode = mode;
    LinearQuery without = q;
    without.workspace_attached = false;
    without.workspace_bytes = 0;
    if (choose_linear(q, -1).cfg != choose_linear(without, -1).cfg) return q.workspace_bytes;
  }
  return 0;
}

}  // namespace
}  // namespace tmq

TMQ_EXPORT int64_t tmq_linear_scratch_bytes(int64_t M, int64_t N, int64_t K, int on_grid) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (K % 16 == 0 && on_grid) return split_bytes_used(M, N, K);
  if (wloop_ragged_tile(M, N, K) != 0 && !wloop_ragged_copied(M, N, K)) return 0;
  if ((M <= kDecodeRowsAuto && K >= 16) || (ragged_route(M, N, K, false, true) != RaggedTile::kCopy && ragged_route(M, N, K, true, true) != RaggedTile::kCopy) || !regrid_limits_ok(M, K)) return 0;
  return regrid_bytes(M, K) + split_bytes_used(M, N, regrid_pitch(K));
}

TMQ_EXPORT int tmq_linear_rows_in_place(int64_t M, int64_t N, int64_t K) {
  return M > 0 && N > 0 && wloop_ragged_tile(M, N, K) != 0 && !few_rows_copied(M, N, K) ? 1 : 0;
}

TMQ_EXPORT int tmq_linear_split_plan(int64_t M, int64_t N, int64_t K, int32_t* splits, int32_t* stages) {
  if (M < 0 || N < 0 || K < 0 || splits == nullptr || stages == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  const SplitPlan p = (M > 0 && N > 0 && K > 0) ? plan_split(M, N, K) : SplitPlan{};
  *splits = p.splits;
  *stages = p.stages;
  return TMQ_OK;
}

static_assert(sizeof(tmq_linear_choice) == 48, "tmq_linear_choice layout changed");

TMQ_EXPORT int tmq_linear_kernel_choice(int64_t M, int64_t N, int64_t K, int64_t ldx, int32_t flags,
                                        int32_t forced_kernel, int32_t compute_units, tmq_linear_choice* out) {
  if (out == nullptr || M < 0 || N < 0 || K < 0 || ldx < K || (flags & 3) == 3 || compute_units < 0)
    return TMQ_ERR_INVALID_ARGUMENT;
  *out = tmq_linear_choice{};
  out->splits = 1;
  out->k_stages = ceil_div(K, kBK);
  if (M == 0 || N == 0) return TMQ_OK;  // nothing is launched
  LinearQuery q;
  q.M = M;
  q.N = N;
  q.K = K;
  q.ldx = ldx;
  q.mode = (flags & 3) == TMQ_LINEAR_OUT_F32 ? kOutF32 : (flags & 3) == TMQ_LINEAR_OUT_ACC32 ? kOutAcc32 : kOutU8;
  q.vec_ok = (flags & 8) == 0 && K >= 16 && K % 16 == 0 && ldx % 16 == 0;
  q.workspace_attached = (flags & 4) != 0;
  q.workspace_bytes = q.workspace_attached && K > 0 ? split_workspace_bytes(plan_split(M, N, K), M) : 0;
  const LinearChoice c = choose_linear(q, forced_kernel - 1);
  if (c.cfg == kNoKernel) return TMQ_OK;
  int bm = 0, bn = 0, waves = 4;
  switch (c.cfg) {
    case 0: bm = 256, bn = 256; break;
    case 3: case 6: case 20: bm = 256, bn = 256, waves = 8; break;
    case 1: case 13: bm = 128, bn = 128; break;
    case 7: bm = 128, bn = 128, waves = ceil_div(M, 128) * ceil_div(N, 128) <= 256 ? 8 : 4; break;
    case 2: bm = 64, bn = 64, waves = 4 * c.groups; break;
    case 21: bm = 64, bn = 64; break;
    case 14: bm = 64, bn = 64, waves = 8; break;
    case 4: bm = 128, bn = 256; break;
    case 17: case 19: bm = 128, bn = 256, waves = 8; break;
    case 5: bm = 256, bn = 128; break;
    case 22: bm = 128, bn = 64; break;
    case 23: bm = 64, bn = 128, waves = c.onepass ? 8 : 4; break;
    case 24: bm = 32, bn = 32; break;
    case 25: bm = 32, bn = 32, waves = kWloopWaves; break;
    case 26: bm = 32, bn = 64, waves = 8; break;
    case 27: bm = 64, bn = 64, waves = 8; break;
    case 29: bm = 32, bn = 32, waves = kWloopWaves; break;
    case 30: bm = 32, bn = 64, waves = kWloopWaves; break;
    case 8: bm = 16 * static_cast<int>(ceil_div(M, 16)), bn = 16, waves = kDecodeWaves; break;
    case 28: bm = 16 * static_cast<int>(ceil_div(M, 16)), bn = 16, waves = resident_pair(M, N, K, compute_units) ? 8 : kResidentWaves; break;
    default: break;  // 9: one thread per four outputs
  }
  out->kernel = c.cfg + 1;
  out->tile_rows = bm;
  out->tile_channels = bn;
  out->waves = waves;
  out->splits = c.split.splits;
  out->split_stages = c.split.stages;
  if (c.cfg == 9) {
    out->tiles = out->blocks = ceil_div(M * ceil_div(N, 4), 256);
  } else {
    out->tiles = ceil_div(M, bm) * ceil_div(N, bn) * c.split.splits;
    out->blocks = out->tiles;
    if (c.cfg == 20 && out->tiles > compute_units) out->blocks = compute_units / 8 * 8;
    if (c.cfg == 25 && wstream_pairs(M, N)) out->blocks = ceil_div(M, 32) * ceil_div(N, 64);
    if (c.cfg == 28) out->blocks = std::min<int64_t>(out->tiles, (waves == 8 ? 2 : 1) * static_cast<int64_t>(compute_units));
  }
  return TMQ_OK;
}

namespace tmq {
namespace {

// quantized::linear with the split-K scratch passed beside the descriptor.
int linear_u8s8(const tmq_linear_desc* d, void* workspace, int64_t workspace_bytes, tmq_stream_t stream) {
  GemmArgs a{};
  XLinear xs{};
  bool vec_ok = false;
  const int rc = fill_args(d, &a, &xs, &vec_ok);
  if (rc != TMQ_OK || d->M == 0 || d->N == 0) return rc;
  if (d->y == nullptr || d->w_scales == nullptr || d->ldy < d->N) return TMQ_ERR_INVALID_ARGUMENT;
  if (!(d->x_scale > 0.f) || !(d->out_scale > 0.f)) return TMQ_ERR_INVALID_ARGUMENT;
  const int qmin = d->out_signed ? -128 : 0, qmax = d->out_signed ? 127 : 255;
  if (d->out_zero_point < qmin || d->out_zero_point > qmax) return TMQ_ERR_INVALID_ARGUMENT;
  a.w_scales = d->w_scales;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.bias = d->bias;
  a.acc_coef = (d->x_signed ? 0 : 128) - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.out_scale = d->out_scale;
  a.zp_f = static_cast<float>(d->out_zero_point);
  a.lo_f = static_cast<float>(d->relu ? d->out_zero_point : qmin);
  a.hi_f = static_cast<float>(qmax);
  a.y = d->y;
  a.ldy = d->ldy;
  hipStream_t s = as_stream(stream);
  return d->out_signed
             ? dispatch_linear<kOutS8>(a, xs, d->x_signed, vec_ok, d->kernel - 1, s, workspace, workspace_bytes)
             : dispatch_linear<kOutU8>(a, xs, d->x_signed, vec_ok, d->kernel - 1, s, workspace, workspace_bytes);
}

}  // namespace
}  // namespace tmq

TMQ_EXPORT int tmq_linear(const tmq_linear_desc* d, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  return linear_u8s8(d, d->workspace, d->workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// quantized::linear for callers that cannot allocate: the split-K partial sums
// go to a fixed array in the library's own device memory.
// ---------------------------------------------------------------------------
namespace tmq {
namespace {

// Every split plan fits: splits x tiles <= 256 blocks of 128 x 128 int32 sums.
constexpr int64_t kStaticWorkspaceBytes = int64_t{16} << 20;
static_assert(kStaticWorkspaceBytes == TMQ_LINEAR_STATIC_WORKSPACE_BYTES, "header and library disagree");
static __device__ __align__(256) uint8_t scratch[kStaticWorkspaceBytes];

// Device address of `scratch` on every device used so far.  The array's name
// is a host-side handle in host code; each device holds its own copy of the
// array at its own address, which hipGetSymbolAddress reports for the current
// device.  Two threads that race on a device's first call store the same value.
std::atomic<void*> g_scratch_addr[kMaxDevices];

// The array of the device that owns `s` -- which must be the current device: the
// symbol's address can only be asked for on the current device.
int static_workspace(hipStream_t s, void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return TMQ_ERR_LAUNCH;
  if (s != nullptr) {
    int sdev = -1;
    if (hipStreamGetDevice(s, &sdev) != hipSuccess) {
      (void)hipGetLastError();
      return TMQ_ERR_INVALID_ARGUMENT;
    }
    if (sdev != dev) return TMQ_ERR_INVALID_ARGUMENT;  // another GPU's stream: that GPU has its own array
  }
  void* p = g_scratch_addr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return TMQ_ERR_LAUNCH;
    g_scratch_addr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return TMQ_OK;
}

}  // namespace
}  // namespace tmq

TMQ_EXPORT int tmq_linear_static_workspace(const tmq_linear_desc* d, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->M < 0 || d->N < 0 || d->K < 0) return TMQ_ERR_INVALID_ARGUMENT;
  const int64_t need = (d->M > 0 && d->N > 0 && d->K > 0) ? split_workspace_bytes(plan_split(d->M, d->N, d->K), d->M) : 0;
  if (need > kStaticWorkspaceBytes) return TMQ_ERR_WORKSPACE;  // the caller's own workspace and tmq_linear then
  void* ws = nullptr;
  if (need > 0) {
    const int rc = static_workspace(as_stream(stream), &ws);
    if (rc != TMQ_OK) return rc;
  }
  return linear_u8s8(d, ws, need, stream);
}

TMQ_EXPORT int tmq_linear_acc32(const tmq_linear_desc* d, int32_t* acc, int64_t ldacc,
                                tmq_stream_t stream) {
  GemmArgs a{};
  XLinear xs{};
  bool vec_ok = false;
  const int rc = fill_args(d, &a, &xs, &vec_ok);
  if (rc != TMQ_OK || d->M == 0 || d->N == 0) return rc;
  if (acc == nullptr || ldacc < d->N) return TMQ_ERR_INVALID_ARGUMENT;
  a.acc_coef = d->x_signed ? 0 : 128;  // undo the x ^ 0x80 shift only
  a.y = acc;
  a.ldy = ldacc;
  return dispatch_linear<kOutAcc32>(a, xs, d->x_signed, vec_ok, d->kernel - 1, as_stream(stream), d->workspace,
                                    d->workspace_bytes);
}

TMQ_EXPORT int tmq_linear_float(const tmq_linear_desc* d, const tmq_qparams* x_qparams_dev, void* y, int64_t ldy,
                                int kind, tmq_stream_t stream) {
  if (kind != TMQ_FLOAT_F32 && kind != TMQ_FLOAT_BF16 && kind != TMQ_FLOAT_F16) return TMQ_ERR_INVALID_ARGUMENT;
  GemmArgs a{};
  XLinear xs{};
  bool vec_ok = false;
  const int rc = fill_args(d, &a, &xs, &vec_ok);
  if (rc != TMQ_OK || d->M == 0 || d->N == 0) return rc;
  if (y == nullptr || d->w_scales == nullptr || ldy < d->N) return TMQ_ERR_INVALID_ARGUMENT;
  if (x_qparams_dev == nullptr && !(d->x_scale > 0.f)) return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(y, kind == TMQ_FLOAT_F32 ? 4 : 2)) return TMQ_ERR_ALIGNMENT;
  a.f_kind = kind;
  a.w_scales = d->w_scales;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.bias = d->bias;
  a.acc_base = d->x_signed ? 0 : 128;
  a.acc_coef = a.acc_base - d->x_zero_point;
  a.x_scale = d->x_scale;
  a.x_qp_dev = x_qparams_dev;
  a.out_scale = 1.f;
  a.lo_f = d->relu ? 0.f : -__builtin_inff();
  a.y = y;
  a.ldy = ldy;
  return dispatch_linear<kOutF32>(a, xs, d->x_signed, vec_ok, d->kernel - 1, as_stream(stream), d->workspace,
                                  d->workspace_bytes);
}

TMQ_EXPORT int tmq_linear_f32(const tmq_linear_desc* d, const tmq_qparams* x_qparams_dev, float* y,
                              int64_t ldy, tmq_stream_t stream) {
  return tmq_linear_float(d, x_qparams_dev, y, ldy, TMQ_FLOAT_F32, stream);
}

// The float rows of the one-launch dynamic linear as the resident kernel holds them: 16 waves x 64 lanes x up to 16 groups of
// four values.  More than 8 groups only against many channels, whose stream is what the block's work on the rows passes under.
// One launch over two, each queued behind the one before, of 16 x 2560, 9 x 4096, 16 x 4096, 12 x 5120, 8 x 8192, 5 x 8192 and 14 x 3000,
// whose rows are off the 16-byte grid: N = 4096 0.97, 0.97, 1.06, 0.94, 1.01, 1.00, 0.91; 6144 0.95, 0.95, 0.97, 0.94, 0.92, 0.96, 0.87;
// 8192 0.91, 1.04, 0.95, 0.95, 0.99, 1.04, 0.87; 10240 0.90, 0.92, 0.92, 0.93, 0.95, 0.94, 0.84; 12288 0.92, 0.93, 0.94, 0.94, 0.99, 0.96,
// 0.85; 16384 0.96, 0.96, 0.95, 0.97, 0.96, 0.95, 0.84; 24576 0.97, 1.00, 0.98, 0.96, 0.95, 0.95, 0.78 (16 x 4096 -> 10240 15.3 | 14.0 us).
// From 10240 on never behind, below by up to 6 %; the line follows N, not the weights' bytes (5 x 8192 -> 8192, 64 Mi: 1.04; 16 x 2560 ->
// 10240, 25 Mi: 0.90).
constexpr int64_t kDynResidentMaxValues = 32768, kDynResidentMostValues = 65536, kDynResidentManyChannels = 10240;

namespace {
// Groups of four values, the last one of a row perhaps partly behind its end.
int64_t dyn_groups(int64_t M, int64_t K) { return M * ceil_div(K, 4); }
bool dyn_resident_ok(int64_t M, int64_t N, int64_t K, int cus) {
  return 4 * dyn_groups(M, K) <= (N < kDynResidentManyChannels ? kDynResidentMaxValues : kDynResidentMostValues) &&
         resident_limits_ok(M, N, round_up(K, 16), K, cus);
}
}  // namespace

TMQ_EXPORT int tmq_linear_dynamic_small_takes(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || M > 16 || N < 1 || K < 16 || ceil_div(N, 16) > 0x7fffffff) return 0;
  if (4 * dyn_groups(M, K) <= kDynSmallMaxValues) return 1;
  const int cus = cu_count();
  return dyn_resident_ok(M, N, K, cus > 0 ? cus : 256) ? 1 : 0;
}

namespace tmq {
namespace {

constexpr int64_t kDynTilesMaxK = 2048;
// Channels per tile of the one-launch dynamic linear of more than 16 rows, 0: not such a shape.  All its blocks have to be on the chip
// together (one that waits for a block behind it finds that one's range itself, but late): one a CU, two up to K = 512, where
// their registers and LDS allow that (us, two launches | 64 channels on 257 to 512 tiles: 135 x 64 -> 5104 7.8 | 6.1, 79 x 263 -> 10799
// 9.6 | 7.0, 3041 x 256 -> 184 8.5 | 6.6, 2825 x 448 -> 296 10.2 | 8.2; 32 channels there, where 64 have one a CU, 3370 x 344 -> 111 7.5
// against 5.9).
int dyn_tile(int64_t M, int64_t N, int64_t K) {
  if (M <= 16 || M > 32 * kRangeParts || N <= 0 || N >= (int64_t{1} << 29) || K < 16 || K > kDynTilesMaxK) return 0;
  const int64_t tiles_m = ceil_div(M, 32), cus = cu_count() > 0 ? cu_count() : 256;
  return tiles_m * ceil_div(N, 32) <= cus ? 32 : tiles_m * ceil_div(N, 64) <= (K <= 512 ? 2 * cus : cus) ? 64 : 0;
}
template <int CT>
auto dyn_tiles_kernel(int64_t K) {
  return K <= 256    ? linear_dynamic_tiles_kernel<CT, 32>
         : K <= 512  ? linear_dynamic_tiles_kernel<CT, 64>
         : K <= 1024 ? linear_dynamic_tiles_kernel<CT, 128>
                     : linear_dynamic_tiles_kernel<CT, 256>;
}

}  // namespace
}  // namespace tmq

TMQ_EXPORT int64_t tmq_linear_dynamic_tiles_workspace(int64_t M, int64_t N, int64_t K) {
  return dyn_tile(M, N, K) == 0 ? -1 : M <= 32 ? 0 : ceil_div(M, 32) * static_cast<int64_t>(sizeof(v4u));
}

TMQ_EXPORT int tmq_linear_dynamic_tiles(const tmq_linear_desc* d, const float* x, int64_t ldx, int reduce_range, float* y,
                                        int64_t ldy, int polls, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  const int tile = dyn_tile(d->M, d->N, d->K);
  if (tile == 0) return TMQ_ERR_UNSUPPORTED;
  if (x == nullptr || y == nullptr || d->w_packed == nullptr || d->w_colsum == nullptr || d->w_scales == nullptr || ldx < d->K ||
      ldy < d->N)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(x, 4) || !aligned(d->w_packed, 16) || !aligned(y, 4)) return TMQ_ERR_UNSUPPORTED;
  hipStream_t s = as_stream(stream);
  const int64_t tiles_m = ceil_div(d->M, 32), tiles_n = ceil_div(d->N, tile);
  if (tiles_m > 1 && (d->workspace == nullptr || d->workspace_bytes < tiles_m * static_cast<int64_t>(sizeof(v4u)) ||
                      !aligned(d->workspace, 16) || replayed(s)))
    return TMQ_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.M = d->M;
  a.N = d->N;
  a.K = d->K;
  a.w_packed = static_cast<const uint8_t*>(d->w_packed);
  a.w_kchunks = packed_kchunks(d->K);
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.bias = d->bias;
  a.lo_f = d->relu ? 0.f : -__builtin_inff();
  a.y = y;
  a.ldy = ldy;
  const bool by_rows = 4 * d->M >= d->N;
  const int64_t minor = by_rows ? tiles_n : tiles_m;
  const DynTileOrder order{static_cast<uint32_t>(tiles_m), static_cast<uint32_t>(tiles_n),
                           minor == 1 ? 0u : static_cast<uint32_t>(((int64_t{1} << 32) + minor - 1) / minor), by_rows ? 1 : 0};
  const RangeWords range{static_cast<v4u*>(d->workspace), tiles_m > 1 ? next_range_tag() : 0, polls < 0 ? kRangePolls : polls};
  enqueue(tile == 32 ? dyn_tiles_kernel<1>(d->K) : dyn_tiles_kernel<2>(d->K), dim3(static_cast<unsigned>(tiles_m * tiles_n)),
          dim3(kDynTileThreads), 0, s, a, x, ldx, reduce_range, range, order);
  return launch_status();
}

TMQ_EXPORT int tmq_linear_dynamic_small(const tmq_linear_desc* d, const float* x, int64_t ldx, int reduce_range,
                                        float* y, int64_t ldy, tmq_stream_t stream) {
  if (d == nullptr) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->M < 0 || d->N < 0 || d->K < 0) return TMQ_ERR_INVALID_ARGUMENT;
  if (d->M == 0 || d->N == 0) return TMQ_OK;
  if (d->M > 16 || d->K < 16) return TMQ_ERR_UNSUPPORTED;
  if (x == nullptr || y == nullptr || d->w_packed == nullptr || d->w_colsum == nullptr || d->w_scales == nullptr)
    return TMQ_ERR_INVALID_ARGUMENT;
  if (ldx < d->K || ldy < d->N) return TMQ_ERR_INVALID_ARGUMENT;
  if (!aligned(x, 4) || !aligned(d->w_packed, 16) || !aligned(y, 4)) return TMQ_ERR_UNSUPPORTED;
  const int64_t blocks = ceil_div(d->N, 16);
  if (blocks > 0x7fffffff) return TMQ_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.M = d->M;
  a.N = d->N;
  a.K = d->K;
  a.w_packed = static_cast<const uint8_t*>(d->w_packed);
  a.w_kchunks = packed_kchunks(d->K);
  a.colsum = d->w_colsum;
  a.w_scales = d->w_scales;
  a.w_scale_stride = d->w_per_channel ? 1 : 0;
  a.bias = d->bias;
  a.lo_f = d->relu ? 0.f : -__builtin_inff();
  a.y = y;
  a.ldy = ldy;
  hipStream_t s = as_stream(stream);
  // Two kernels: a block per 16 channels that repeats the work on the input (up to 16384 values), and
  // one block per CU that does it once for all its channel groups (dyn_resident_ok).
  // desc->kernel pins one for tests: 9 the first, 29 the second.
  const int cus = cu_count();
  const bool resident_ok = dyn_resident_ok(d->M, d->N, d->K, cus);
  const bool small_ok = 4 * dyn_groups(d->M, d->K) <= kDynSmallMaxValues;
  if ((d->kernel == 9 && !small_ok) || (d->kernel == 29 && !resident_ok) || (!small_ok && !resident_ok))
    return TMQ_ERR_UNSUPPORTED;
  const bool resident =
      resident_ok && (d->kernel == 29 || (d->kernel != 9 && (!small_ok || dynamic_resident_preferred(d->M, d->N, d->K))));
  if (resident) {
    const XLinear none{nullptr, 0};
    const dim3 grid(static_cast<unsigned>(blocks < cus ? blocks : cus)), block(kResidentThreads);
    const int64_t held = ceil_div(dyn_groups(d->M, d->K), kResidentThreads);  // float4 per thread
    if (held <= 2)
      enqueue(linear_resident_kernel<kOutF32, 1, kResidentWaves, 2>, grid, block, 0, s, a, none, x, ldx, reduce_range);
    else if (held <= 4)
      enqueue(linear_resident_kernel<kOutF32, 1, kResidentWaves, 4>, grid, block, 0, s, a, none, x, ldx, reduce_range);
    else if (held <= 8)
      enqueue(linear_resident_kernel<kOutF32, 1, kResidentWaves, 8>, grid, block, 0, s, a, none, x, ldx, reduce_range);
    else
      enqueue(linear_resident_kernel<kOutF32, 1, kResidentWaves, 16>, grid, block, 0, s, a, none, x, ldx, reduce_range);
    return launch_status();
  }
  const size_t lds = static_cast<size_t>(d->M) * static_cast<size_t>(round_up(d->K, 16) + 16);
  const dim3 grid(static_cast<unsigned>(blocks)), block(kDecodeWaves * kWave);
  const int64_t groups = ceil_div(dyn_groups(d->M, d->K), kDecodeWaves * kWave);  // float4 per thread
  if (groups <= 1)
    enqueue(linear_decode_dynamic_kernel<1>, grid, block, lds, s, a, x, ldx, reduce_range);
  else if (groups <= 2)
    enqueue(linear_decode_dynamic_kernel<2>, grid, block, lds, s, a, x, ldx, reduce_range);
  else if (groups <= 4)
    enqueue(linear_decode_dynamic_kernel<4>, grid, block, lds, s, a, x, ldx, reduce_range);
  else
    enqueue(linear_decode_dynamic_kernel<8>, grid, block, lds, s, a, x, ldx, reduce_range);
  return launch_status();
}
