// Values that a kernel hands to the host before it ends (device code).
#pragma once

#include "common.h"

namespace tmq {
namespace {

// What the host waits for goes to it as one or two 8-byte words in pinned host memory, a
// ticket in the upper half and the payload in the lower one: each word is a single store,
// so the host needs no order between them and the device no fence (a system-scope release
// would write back the L2s first).
__device__ __forceinline__ void report_word(uint64_t* word, uint32_t ticket, uint32_t payload) {
  __hip_atomic_store(word, (static_cast<uint64_t>(ticket) << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
struct RangeReport {
  tmq_host_report* to;
  uint32_t ticket;
  uint32_t slot;  // below TMQ_HOST_REPORTS, this report's own among the calls in flight
};
__device__ __forceinline__ void report_range(const RangeReport& r, float mn, float mx) {
  if (r.to == nullptr) return;
  report_word(&r.to->word[0], r.ticket, __builtin_bit_cast(uint32_t, mn));
  report_word(&r.to->word[1], r.ticket, __builtin_bit_cast(uint32_t, mx));
}

}  // namespace
}  // namespace tmq
