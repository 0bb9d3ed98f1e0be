// What the host asks a device once (host code).
#pragma once

#include <atomic>

#include "common.h"

namespace tmq {
namespace {

constexpr int kMaxDevices = 64;

// Compute units of the current device (cached per device; two threads that race
// on a device's first call store the same value).
inline int cu_count() {
  static std::atomic<int> cache[kMaxDevices];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cache[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace
}  // namespace tmq
