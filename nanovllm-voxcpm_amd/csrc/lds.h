// Host side: LDS beyond 64 KB per workgroup.  The runtime wants it allowed per kernel and per device.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>

namespace mlora {

constexpr int kPlainLds = 64 * 1024, kMostLds = 160 * 1024;

// Lets launches of Kernel on the calling thread's current device take `bytes` of dynamic LDS.
template <auto Kernel> void allow_lds(int bytes) {
  if (bytes <= kPlainLds) return;
  static std::atomic<uint64_t> allowed{0};  // bit per device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return;  // (the launch reports it)
  const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;
  if (bit & allowed.load(std::memory_order_relaxed)) return;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds) == hipSuccess)
    allowed.fetch_or(bit, std::memory_order_relaxed);
}

}  // namespace mlora
