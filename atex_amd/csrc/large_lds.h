// Dynamic LDS beyond the default limit of a launch.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include "plan.h"

namespace atexn {

// The kernels that keep a row (or its accumulators, or a slab) in LDS ask for more dynamic LDS than
// a launch gets by default: the limit is raised once per kernel and device.
template <auto Kernel>
inline hipError_t allow_large_lds() {
  static std::atomic<uint64_t> done{0};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    dev = -1;
  }
  if (dev >= 0 && ((done.load(std::memory_order_acquire) >> dev) & 1)) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(kPlanLdsBytes - kPlanBwdLdsReserve));
  if (e == hipSuccess && dev >= 0) done.fetch_or(uint64_t(1) << dev, std::memory_order_release);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

}  // namespace atexn
