// Range, parameters and codes of a dynamic quantization in one launch (device code for gfx950 only).
#pragma once

#include <limits>

#include "common.h"
#include "host_report.h"
#include "qparams.h"
#include "range_exchange.h"

namespace tmq {
namespace {

// At most one block per CU reads its part of the input into registers, tells the others its range, waits for theirs and
// converts what it holds: the input is read once, and neither a second launch nor its first reads lie between range and
// codes.  256 CUs have 128 MB of registers; 32 groups of four values a thread are 64 MB of them, 16 Mi values.  Parts
// beyond that are read again, from the last-level cache while it has them.
//
// What bounds it: up to a million values the exchange of the ranges (about 1.5 us: one store past the L2, one read of 4 KB
// that every block repeats until it is complete) and the launch; then memory.  A call after the other on the stream, range
// pass and quantizer as two launches | this, us: 64 Ki values 4.8 | 3.9 (there against the one launch whose blocks all read
// everything), 128 Ki 5.4 | 3.9, 1 Mi 5.8 | 4.4, 1912 x 3392 13.2 | 8.7, 1507 x 8160 19.2 | 12.2, 4096 x 4096 26.8 | 15.0 ... 17.5,
// 4096 x 8192 51 | 41; 16 Mi values from memory are 10.3 us at 6.5 TB/s.  Blocks of 512 threads: of 256, 512 and 1024, 1 to
// 16 % ahead from 64 Ki values on (1024 threads have no registers left for 16 groups: 22.5 against 19.5).  Codes leave past the
// L2s (19.5 -> 18.1 at 4096 x 4096, level below a million values).  From 24 groups on the input is read past the caches: it
// is not read twice, and the caches are left to what is (4096 x 4096 18.1 -> 15.0 ... 17.5; 16 groups and fewer measured slower
// that way when the same input comes again, 9.2 -> 9.4).
constexpr int kHeldThreads = 512;
constexpr int kHeldBlocks = kRangeParts;
constexpr int kHeldMost = 32;
constexpr int kHeldStream = 24;

// `total` words of four codes, H + more of them for each thread.  Dense (not ROWS): x on the 16-byte grid, `tail` values
// (below four) behind the last word.  ROWS: rows of K >= 4 values at any 4-byte alignment -> rows of pitch4 words; the codes
// behind a row's end are whatever its last values give.  sign_flip 0x80808080 for signed codes, which FUSED does not have
// (see quantize_four).  The range goes to the host as a whole (report) or, if there are `parts`, each block's own.
template <bool FUSED, bool ROWS, int H>
__global__ __launch_bounds__(kHeldThreads) void dynamic_quantize_held_kernel(
    const float* __restrict__ x, uint32_t* __restrict__ q4, int32_t total, int32_t K, int32_t pitch4, int32_t tail,
    RangeWords range, int32_t more, uint32_t sign_flip, int qmin, int qmax, int reduce_range, tmq_qparams* __restrict__ out,
    RangeReport report, uint64_t* parts) {
  constexpr int kWaves = kHeldThreads / kWave;
  constexpr int kRepairAhead = 4;
  constexpr int kAhead = H >= 16 ? 16 : 4;  // (of the words that are not held; only H = kHeldMost has any)
  __shared__ float s_range[2 * kWaves], s_inv, s_zp;
  __shared__ int s_missing;
  const int t = threadIdx.x, own = static_cast<int>(blockIdx.x), blocks = static_cast<int>(gridDim.x);
  const int step = blocks * kHeldThreads;
  // a thread's words: its first, then one every `step`
  struct Place {
    int i, row, c4;
  };
  const int step_rows = ROWS ? step / pitch4 : 0, step_c4 = ROWS ? step - step_rows * pitch4 : 0;
  const auto place = [&](int block) {
    Place p{block * kHeldThreads + t, 0, 0};
    if (ROWS) {
      p.row = p.i / pitch4;
      p.c4 = p.i - p.row * pitch4;
    }
    return p;
  };
  const auto advance = [&](Place& p) {
    p.i += step;
    if (ROWS) {
      p.row += step_rows;
      p.c4 += step_c4;
      if (p.c4 >= pitch4) {
        p.c4 -= pitch4;
        ++p.row;
      }
    }
  };
  // The four values of a word (words past the end: of one inside; a row's last word: the row's last four).
  const auto load = [&](const Place& p) -> v4f {
    if (ROWS) {
      const bool in = p.i < total;
      const int c = in ? 4 * p.c4 : 0;
      return reinterpret_cast<const FourFloats*>(x + static_cast<int64_t>(in ? p.row : 0) * K + (c + 4 <= K ? c : K - 4))->v;
    }
    const v4f* src = reinterpret_cast<const v4f*>(x) + (p.i < total ? p.i : total - 1);
    return H >= kHeldStream ? __builtin_nontemporal_load(src) : *src;
  };
  const auto take_tail = [&](int block, float& mn, float& mx) {
    if (!ROWS && block == 0 && t < tail) {
      const float v = x[4 * static_cast<int64_t>(total) + t];
      mn = fminf(mn, v);
      mx = fmaxf(mx, v);
    }
  };
  // The range of a block's part, to where all blocks see it (and to the host).
  const auto publish = [&](int block, float& mn, float& mx, uint64_t* part) {
    block_range<kWaves>(mn, mx, s_range, t);
    if (t == 0) {
      put_range(range, block, mn, mx);
      if (part != nullptr)  // (one store of eight bytes: complete or not there)
        __hip_atomic_store(part, (static_cast<uint64_t>(__builtin_bit_cast(uint32_t, mx)) << 32) | __builtin_bit_cast(uint32_t, mn),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  };

  float mn = std::numeric_limits<float>::infinity();
  float mx = -std::numeric_limits<float>::infinity();
  Place at = place(own);
  if (H == kHeldMost && more > 0) {
    Place p = at;
    for (int u = 0; u < H; ++u) advance(p);
    for (int u = 0; u < more; u += kAhead) {
      v4f v[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        v[j] = load(p);
        advance(p);
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) take_four(v[j], mn, mx);
    }
  }
  v4f held[H];
#pragma unroll
  for (int u = 0; u < H; ++u) {
    held[u] = load(at);
    advance(at);
  }
#pragma unroll
  for (int u = 0; u < H; ++u) take_four(held[u], mn, mx);
  take_tail(own, mn, mx);
  publish(own, mn, mx, parts == nullptr ? nullptr : parts + own);

  // All ranges, and the parameters from them.
  RangeView view(blocks);
  for (int polls = range.polls;; polls = 0) {
    if (t < kWave) {
      const int missing = get_ranges(range, blocks, own, polls, view, mn, mx);
      if (missing < 0) {
        if (own == 0 && t == 0) report_range(report, mn, mx);
        double s;
        int32_t z;
        choose_qparams(mn, mx, qmin, qmax, reduce_range != 0, &s, &z);
        if (t == 0) {
          if (own == 0) {
            out->scale = s;
            out->zero_point = z;
            out->reserved = 0;
          }
          s_inv = 1.0f / static_cast<float>(s);  // IEEE division, as in resolve()
          s_zp = static_cast<float>(z);
        }
      }
      if (t == 0) s_missing = missing;
    }
    __syncthreads();
    const int missing = s_missing;
    if (missing < 0) break;
    // That block has not run yet -- the chip is not this launch's alone -- or not for this long.
    float a = std::numeric_limits<float>::infinity();
    float b = -std::numeric_limits<float>::infinity();
    Place p = place(missing);
#pragma unroll 1
    for (int u = 0; u < H + more; u += kRepairAhead) {  // (past the part's end: of another one, or the last word again)
      v4f v[kRepairAhead];
#pragma unroll
      for (int j = 0; j < kRepairAhead; ++j) {
        v[j] = load(p);
        advance(p);
      }
#pragma unroll
      for (int j = 0; j < kRepairAhead; ++j) take_four(v[j], a, b);
    }
    take_tail(missing, a, b);
    publish(missing, a, b, nullptr);
    if (t < kWave) view.add(missing, a, b);
    __syncthreads();
  }

  const float inv = s_inv, zp_f = s_zp;
  const float zp_u = sign_flip != 0 ? zp_f + 128.f : zp_f;
  const auto code = [&](float v, int j, uint32_t packed) {
    const float r = FUSED ? __builtin_fmaf(v, inv, zp_f) : __builtin_rintf(v * inv) + zp_u;
    return __builtin_amdgcn_cvt_pk_u8_f32(r, j, packed);
  };
  const auto store = [&](const Place& p, v4f v) {
    if (p.i >= total) return;
    if (ROWS) {
      const int d = 4 * p.c4 + 4 - K;  // a row's last word holds the row's last four values
      if (d > 0) {
        v.x = d == 1 ? v.y : d == 2 ? v.z : v.w;
        v.y = d == 1 ? v.z : v.w;
        v.z = v.w;
      }
    }
    uint32_t packed = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) packed = code(v[j], j, packed);
    st4_through(&q4[p.i], packed ^ sign_flip);
  };
  at = place(own);
#pragma unroll
  for (int u = 0; u < H; ++u) {
    store(at, held[u]);
    advance(at);
  }
  if (H == kHeldMost) {
    for (int u = 0; u < more; u += kAhead) {
      v4f v[kAhead];
      Place p = at;
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        v[j] = load(at);
        advance(at);
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        store(p, v[j]);
        advance(p);
      }
    }
  }
  if (!ROWS && own == 0 && t < tail) {
    const int64_t i = 4 * static_cast<int64_t>(total) + t;
    reinterpret_cast<uint8_t*>(q4)[i] = static_cast<uint8_t>(code(x[i], 0, 0u) ^ (sign_flip & 0xffu));
  }
}

}  // namespace
}  // namespace tmq
