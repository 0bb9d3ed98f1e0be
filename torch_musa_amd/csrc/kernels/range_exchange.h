// The blocks of one launch tell each other the minimum and maximum of their parts of the input.
#pragma once

#include <atomic>
#include <chrono>
#include <limits>

#include "absent_parts.h"
#include "common.h"
#include "dynamic_rows.h"
#include "stores_through.h"

namespace tmq {

// A word of 16 bytes for each part, {minimum, low half of the tag, maximum, high half of the tag}.  Either half of a word is
// whole if its half of the tag is this launch's; no other launch of the process has that tag, so what the memory held before
// need not be cleared.  Whoever has read a part may write its word, which says the same whoever does: a block that does not see
// a word in time reads that part itself and remembers it, and so every block ends whether or not the others run beside it.
// Blocks that wait for the same ones read different parts and share what they find (us beside a neighbour that has a quarter | half of
// the CUs to itself for 160 us, each block reading the first absent part behind its own and waiting anew after it | now: quantizing
// 12 Mi values 112, 120 | 45, 50; 16 Mi 124, 131 | 52, 58; 32 Mi 140, 151 | 105, 117; a dynamic linear of 2000 x 2048 -> 250 66, 114 | 39, 48).
// That is still more than launches that need no block beside another one take there (16 Mi values 32, 36; 27 | 16 on an idle chip), and
// beside a kernel on every CU a block waits for as many registers as it holds.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
struct RangeWords {
  v4u* words;
  uint64_t tag;
  int polls;  // of the words, before a block sees to what is missing itself
};
constexpr int kRangeParts = 256;  // at most
// Looks of about a microsecond each, more than the blocks of one launch are apart on an idle chip: from four on level there (16 Mi
// values 16.0 us; two: 23.9), where blocks read again what they do not hold from sixteen on (64 Mi 86.5; eight: 108), hence twice as
// many for those.  Beside a kernel that keeps CUs to itself they are what is waited in vain (16 Mi values with 128 CUs busy for
// 160 us: 4 looks 61, 8 55, 16 58, 32 66 us).
constexpr int kRangePolls = 16;

// What no other launch of this process has: SplitMix64 (Steele, Lea and Flood, "Fast splittable pseudorandom number generators"),
// whose output is a permutation of its counter; the counter's start differs from process to process.
inline uint64_t next_range_tag() {
  static std::atomic<uint64_t> count{static_cast<uint64_t>(std::chrono::steady_clock::now().time_since_epoch().count())};
  uint64_t z = count.fetch_add(1, std::memory_order_relaxed) * 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// A captured launch keeps its arguments: its tag would be in the words already when the graph runs again.
inline bool replayed(hipStream_t s) {
  if (s == nullptr) return false;  // (the null stream cannot be captured)
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;  // unknown: as if it were
}

namespace {

// (one lane)
__device__ __forceinline__ void put_range(const RangeWords& r, int part, float mn, float mx) {
  const v4u word = {__builtin_bit_cast(uint32_t, mn), static_cast<uint32_t>(r.tag), __builtin_bit_cast(uint32_t, mx),
                    static_cast<uint32_t>(r.tag >> 32)};
  st16_through(r.words + part, __builtin_bit_cast(v4i, word));
}

constexpr int kRangeLooks = kRangeParts / kWave;  // words a lane looks at: j kWave + lane

// What a block knows of the others' ranges, kept by its first wave from one look at the words to the next: every look and every
// part that the block reads itself leaves fewer that are absent, whatever happens to the words meanwhile.
struct RangeView {
  uint32_t absent;  // bit j: part j kWave + lane
  float mn, mx;     // of the parts that the lane has seen

  __device__ __forceinline__ explicit RangeView(int parts)
      : absent(0), mn(std::numeric_limits<float>::infinity()), mx(-std::numeric_limits<float>::infinity()) {
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for (int j = 0; j < kRangeLooks; ++j) absent |= (j * kWave + lane < parts ? 1u : 0u) << j;
  }
  // (the block has read this part itself)
  __device__ __forceinline__ void add(int part, float part_mn, float part_mx) {
    if (static_cast<int>(threadIdx.x % kWave) == part % kWave) absent &= ~(1u << (part / kWave));
    mn = fminf(mn, part_mn);
    mx = fmaxf(mx, part_mx);
  }
};

// The range of all `parts`, read by one wave, in all its lanes: -1.  Or, after polls + 1 looks, a part that is not there, another
// one for each `block` (absent_part).
__device__ __forceinline__ int get_ranges(const RangeWords& r, int parts, int block, int polls, RangeView& view, float& mn, float& mx) {
  const int lane = threadIdx.x % kWave;
  for (int poll = 0;; ++poll) {
    v4u w[kRangeLooks];
#pragma unroll
    for (int j = 0; j < kRangeLooks; ++j) {
      const int i = j * kWave + lane;
      if (j * kWave < parts)
        w[j] = __builtin_amdgcn_global_load_b128(
            (__attribute__((address_space(1))) v4u_global*)(r.words + (i < parts ? i : parts - 1)), "agent");
    }
#pragma unroll
    for (int j = 0; j < kRangeLooks; ++j) {
      if (j * kWave >= parts) continue;
      const bool there = w[j].y == static_cast<uint32_t>(r.tag) && w[j].w == static_cast<uint32_t>(r.tag >> 32);
      const uint32_t lo = w[j].x, hi = w[j].z;  // (__builtin_bit_cast of a vector's element takes its first one)
      view.absent &= there ? ~(1u << j) : ~0u;
      view.mn = there ? fminf(view.mn, __builtin_bit_cast(float, lo)) : view.mn;
      view.mx = there ? fmaxf(view.mx, __builtin_bit_cast(float, hi)) : view.mx;
    }
    if (__builtin_amdgcn_ballot_w64(view.absent != 0) == 0) {
      mn = view.mn;
      mx = view.mx;
      wave_minmax_last(mn, mx);
      mn = lane_float(mn, kWave - 1);
      mx = lane_float(mx, kWave - 1);
      return -1;
    }
    if (poll >= polls) break;
    __builtin_amdgcn_s_sleep(1);
  }
  uint64_t absent[kRangeLooks];
#pragma unroll
  for (int j = 0; j < kRangeLooks; ++j) absent[j] = __builtin_amdgcn_ballot_w64((view.absent >> j & 1u) != 0);
  return absent_part(absent, block);
}

// The minimum and maximum that the waves of a block found, in all lanes of its first wave: shared holds 2 W floats; one barrier.
template <int W>
__device__ __forceinline__ void block_range(float& mn, float& mx, float* shared, int t) {
  static_assert(W <= 16 && 16 % W == 0);
  wave_minmax_last(mn, mx);
  if (t % kWave == kWave - 1) {
    shared[t / kWave] = mn;
    shared[W + t / kWave] = mx;
  }
  __syncthreads();
  if (t < kWave) {
    mn = shared[t % W];
    mx = shared[W + t % W];
    row_minmax(mn, mx);
    mn = lane_float(mn, 15);
    mx = lane_float(mx, 15);
  }
}

}  // namespace
}  // namespace tmq
