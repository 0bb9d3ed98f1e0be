// The blocks of one launch tell each other the minimum and maximum of their parts of the input.
#pragma once

#include <atomic>
#include <chrono>
#include <limits>

#include "common.h"
#include "dynamic_rows.h"
#include "stores_through.h"

namespace tmq {

// A word of 16 bytes for each part, {minimum, low half of the tag, maximum, high half of the tag}.  Either half of a word is
// whole if its half of the tag is this launch's; no other launch of the process has that tag, so what the memory held before
// need not be cleared.  Whoever has read a part may write its word, which says the same whoever does: a block that does not see
// a word in time reads that part itself, and so every block ends whether or not the others run beside it.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
struct RangeWords {
  v4u* words;
  uint64_t tag;
  int polls;  // of the words, before a block sees to what is missing itself
};
constexpr int kRangeParts = 256;  // at most
constexpr int kRangePolls = 32;   // of about a microsecond each: more than the blocks of one launch are apart on an idle chip

// What no other launch of this process has (a permutation of a counter; its start differs from process to process).
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

// The range of all `parts`, read by one wave, in all its lanes: -1.  Or, after the last poll, a part that is not there: the next
// one behind `own`, so that blocks that wait together see to different ones.
__device__ __forceinline__ int get_ranges(const RangeWords& r, int parts, int own, float& mn, float& mx) {
  constexpr int kPer = kRangeParts / kWave;
  const int lane = threadIdx.x % kWave;
  uint64_t absent[kPer];
  for (int poll = 0;; ++poll) {
    v4u w[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = j * kWave + lane;
      if (j * kWave < parts)
        w[j] = __builtin_amdgcn_global_load_b128(
            (__attribute__((address_space(1))) v4u_global*)(r.words + (i < parts ? i : parts - 1)), "agent");
    }
    mn = std::numeric_limits<float>::infinity();
    mx = -std::numeric_limits<float>::infinity();
    bool there = true;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      absent[j] = 0;
      if (j * kWave >= parts) continue;
      absent[j] =
          __builtin_amdgcn_ballot_w64(w[j].y != static_cast<uint32_t>(r.tag) || w[j].w != static_cast<uint32_t>(r.tag >> 32));
      there = there && absent[j] == 0;
      const uint32_t lo = w[j].x, hi = w[j].z;  // (__builtin_bit_cast of a vector's element takes its first one)
      mn = fminf(mn, __builtin_bit_cast(float, lo));
      mx = fmaxf(mx, __builtin_bit_cast(float, hi));
    }
    if (there) {
      wave_minmax_last(mn, mx);
      mn = lane_float(mn, kWave - 1);
      mx = lane_float(mx, kWave - 1);
      return -1;
    }
    if (poll >= r.polls) break;
    __builtin_amdgcn_s_sleep(1);
  }
  int first = -1, next = -1;
  for (int j = 0; j < kPer; ++j)
    for (uint64_t m = absent[j]; m != 0; m &= m - 1) {
      int i = j * kWave + __builtin_ctzll(m);
      i = i < parts ? i : parts - 1;
      if (first < 0) first = i;
      if (next < 0 && i > own) next = i;
    }
  return next >= 0 ? next : first;
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
