// Which of the parts that are still missing a block sees to (host and device code).
#pragma once

#include <cstdint>

namespace tmq {

// Bit i % 64 of absent[i / 64]: part i.  The absent part of rank `block` modulo their number, -1 if there is none: blocks next to each
// other take different parts, so that as many are read at a time as there are blocks.  (The first absent part behind a block's own is
// the same one for all blocks where those that run are the first of the grid, as they are beside another stream's kernel.)
template <int WORDS>
constexpr int absent_part(const uint64_t (&absent)[WORDS], int block) {
  int count = 0;
#pragma unroll
  for (int j = 0; j < WORDS; ++j) count += __builtin_popcountll(absent[j]);
  if (count == 0) return -1;
  int rank = block % count, found = -1;
#pragma unroll
  for (int j = 0; j < WORDS; ++j) {
    const int here = __builtin_popcountll(absent[j]);
    if (found < 0 && rank < here) {
      uint64_t left = absent[j];
#pragma unroll 1
      for (int i = 0; i < rank; ++i) left &= left - 1;
      found = 64 * j + __builtin_ctzll(left);
    }
    rank -= here;
  }
  return found;
}

}  // namespace tmq
