#pragma once
#include "gemm_i8_onepass.h"

namespace tmq {

struct KShare {
  uint8_t* words;    // [tiles] 8 bytes
  v4i* partials;     // [tiles][splits][BM * BN / 4]
  uint64_t tag;      // above the low 8 bits
  int splits;
};

constexpr int kShareWaves = 8;
// Tiles of 32 RT rows x 32 CT channels, PB bytes of K a piece; blockIdx.z: which of the runs of pieces.
template <int MODE, int RT, int CT, bool TURN, bool SPLIT, int NW = 8>
__global__ __launch_bounds__(NW* kWave, NW == 8 ? 2 : 2) void gemm_i8_kshare_kernel(GemmArgs a, XLinear xs, KShare ks) {
  constexpr int BM = 32 * RT, BN = 32 * CT, PB = CT * RT == 1 ? 256 : 128, WAVES = NW;
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
  // tiles in runs per XCD, splits of a tile next to each other
  const uint32_t tiles_m = static_cast<uint32_t>(ceil_div(a.M, BM)), tiles_n = static_cast<uint32_t>(ceil_div(a.N, BN));
  const uint32_t id = blockIdx.x, all = gridDim.x;
  const uint32_t share = all / 8, rest = all % 8, xcd = id % 8;
  const uint32_t unit = xcd * share + (xcd < rest ? xcd : rest) + id / 8;
  // order: channel tile, split, row tile
  const uint32_t splits = SPLIT ? static_cast<uint32_t>(ks.splits) : 1u;
  const uint32_t per_n = tiles_m * splits;
  const uint32_t tile_n = __builtin_amdgcn_readfirstlane(unit / per_n);
  const uint32_t in_n = unit - tile_n * per_n;
  const uint32_t split = __builtin_amdgcn_readfirstlane(in_n / tiles_m);
  const uint32_t tile_m = in_n - split * tiles_m;
  const int64_t m0 = static_cast<int64_t>(tile_m) * BM, n0 = static_cast<int64_t>(tile_n) * BN;
  const int K = static_cast<int>(a.K);
  const int KC = K >> 4;                     // 16-byte chunks of a row (K is a multiple of 16)
  const int pieces = (K + PB - 1) / PB;
  // this block's run of pieces
  const int beach = pieces / static_cast<int>(splits), bmore = pieces - beach * static_cast<int>(splits);
  const int bfirst = static_cast<int>(split) * beach + (static_cast<int>(split) < bmore ? static_cast<int>(split) : bmore);
  const int blast = bfirst + beach + (static_cast<int>(split) < bmore ? 1 : 0);
  const int bn = blast - bfirst;
  const int each = bn / WAVES, more = bn - each * WAVES;
  const int first = TURN ? bfirst + wave_u : bfirst + wave_u * each + (wave_u < more ? wave_u : more);
  const int last = TURN ? blast : first + each + (wave_u < more ? 1 : 0);
  constexpr int kNext = TURN ? WAVES : 1;

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
  const auto request = [&](int p, Piece& pc) {
    const int pp = p;
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
  const int64_t n_raw = (n0 + t % BN < a.N ? n0 + t % BN : a.N - 1) + a.n_off;
  const int colsum = a.colsum[n_raw];
  int scale = 0, bias = 0;
  if constexpr (MODE != kOutAcc32) {
    scale = __float_as_int(a.w_scales[n_raw * a.w_scale_stride]);
    bias = __float_as_int((a.bias != nullptr ? a.bias : a.w_scales)[a.bias != nullptr ? n_raw : 0]);
  }
  Piece pc[2];
  v16i acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[rt][ct][r] = 0;

  const auto swizzle = [](int row) { return kLPR == 16 ? row & 15 : (row >> 1) & 7; };
  uint8_t* const mine = &sX[wave_u][0];
  const int flip = static_cast<int>(a.x_xor);
  const auto multiply = [&](int p, Piece& pc) {
    const int c = p * kLPR + slot;
#pragma unroll
    for (int i = 0; i < kNX; ++i) {
      const int r = i * kRPL + lane / kLPR;
      v4i v = pc.x[i];
      const int keep = c < KC ? -1 : 0;
      v = (v ^ v4i{flip, flip, flip, flip}) & v4i{keep, keep, keep, keep};
      *reinterpret_cast<v4i*>(mine + r * PB + ((slot ^ swizzle(r)) << 4)) = v;
    }
    wave_sync_lds();
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const v4i xv = ld16(mine + (32 * rt + li) * PB + (((2 * j + half) ^ swizzle(li)) << 4));
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_i32_32x32x32_i8(pc.w[ct][j], xv, acc[rt][ct], 0, 0, 0);
      }
    }
    wave_sync_lds();
  };
  // (the same number of requests is on its way wherever one is waited for)
  const auto fetch = [&](int p, Piece& into) {
    __builtin_amdgcn_sched_barrier(0);
    request(p, into);
    __builtin_amdgcn_sched_barrier(0);
  };
  int p = first, left = first < last ? (last - first + kNext - 1) / kNext : 0;
  if (left >= 2) {
    fetch(p, pc[0]);
    fetch(p + kNext, pc[1]);
    for (; left >= 4; left -= 2, p += 2 * kNext) {
      multiply(p, pc[0]);
      fetch(p + 2 * kNext, pc[0]);
      multiply(p + kNext, pc[1]);
      fetch(p + 3 * kNext, pc[1]);
    }
    if (left == 3) {
      multiply(p, pc[0]);
      fetch(p + 2 * kNext, pc[0]);
      multiply(p + kNext, pc[1]);
      multiply(p + 2 * kNext, pc[0]);
    } else {
      multiply(p, pc[0]);
      multiply(p + kNext, pc[1]);
    }
  } else if (left == 1) {
    fetch(p, pc[0]);
    multiply(p, pc[0]);
  }
  if (t < BN) {
    s_raw[0][t] = colsum;
    s_raw[1][t] = scale;
    s_raw[2][t] = bias;
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const v4i part = {acc[rt][ct][4 * g], acc[rt][ct][4 * g + 1], acc[rt][ct][4 * g + 2], acc[rt][ct][4 * g + 3]};
      *reinterpret_cast<v4i*>(mine + (32 * rt + li) * kRedPitch + (32 * ct + 8 * g + 4 * half) * 4) = part;
    }
  __syncthreads();
  constexpr int kEach = BM * BN / 4 / (WAVES * kWave) > 0 ? BM * BN / 4 / (WAVES * kWave) : 1;
  if constexpr (!SPLIT) {
#pragma unroll
    for (int idx = t; idx < BM * BN / 4; idx += WAVES * kWave)
      ksplit_finish_four<MODE, BN, WAVES>(a, &sX[0][0], kWaveLds, s_raw, m0, n0, idx);
  } else {
    __shared__ int s_last;
    v4i sum[kEach];
    const uint32_t tile = tile_n * tiles_m + tile_m;
    v4i* const mine_out = ks.partials + (static_cast<int64_t>(tile) * splits + split) * (BM * BN / 4);
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int idx = t + e * WAVES * kWave;
      if (idx < BM * BN / 4) {
        const int row = idx / (BN / 4), cl = (idx % (BN / 4)) * 4;
        v4i s = *reinterpret_cast<const v4i*>(&sX[0][row * kRedPitch + cl * 4]);
#pragma unroll
        for (int w = 1; w < WAVES; ++w) s += *reinterpret_cast<const v4i*>(&sX[w][row * kRedPitch + cl * 4]);
        sum[e] = s;
        st16_through(mine_out + idx, s);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0) {
      uint64_t* const word = reinterpret_cast<uint64_t*>(ks.words) + tile;
      uint64_t old = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), now;
      do {
        now = (old >> 8) == (ks.tag >> 8) ? old + 1 : (ks.tag & ~0xffull) + 1;
      } while (!__hip_atomic_compare_exchange_strong(word, &old, now, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      s_last = (now & 0xff) == splits;
      if (s_last) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    const v4i* const tile_in = ks.partials + static_cast<int64_t>(tile) * splits * (BM * BN / 4);
    constexpr int kAhead = 8;
    for (uint32_t s0 = 0; s0 < splits; s0 += kAhead) {
      v4i v[kAhead][kEach];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int e = 0; e < kEach; ++e) {
          const uint32_t s = s0 + j < splits ? s0 + j : split;
          const int idx = t + e * WAVES * kWave;
          const v4i* src = tile_in + static_cast<int64_t>(s) * (BM * BN / 4) + (idx < BM * BN / 4 ? idx : 0);
          v[j][e] = __builtin_bit_cast(v4i, __builtin_amdgcn_global_load_b128((__attribute__((address_space(1))) v4u_global*)(src), "agent"));
        }
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int e = 0; e < kEach; ++e)
          if (s0 + j < splits && s0 + j != split) sum[e] += v[j][e];
    }
    // over wave 0's partial tile, then as for one block
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int idx = t + e * WAVES * kWave;
      if (idx < BM * BN / 4) {
        const int row = idx / (BN / 4), cl = (idx % (BN / 4)) * 4;
        *reinterpret_cast<v4i*>(&sX[0][row * kRedPitch + cl * 4]) = sum[e];
        ksplit_finish_four<MODE, BN, 1>(a, &sX[0][0], kWaveLds, s_raw, m0, n0, idx);
      }
    }
  }
}

}  // namespace tmq
