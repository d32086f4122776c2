// launch.h -- host-side launch helpers shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace s2 {

// Lets a kernel take up to `bytes` of dynamic LDS.  The attribute belongs to the
// current device's copy of the kernel, so it is set once per device, not once per
// process; `devices` is the kernel's own record of where that was done.
inline hipError_t allow_lds(const void* kernel, uint32_t bytes, std::atomic<uint64_t>& devices) {
  int d = 0;
  hipError_t e = hipGetDevice(&d);
  if (e != hipSuccess) return e;
  const uint64_t bit = uint64_t(1) << (d & 63);
  if (d < 64 && (devices.load(std::memory_order_relaxed) & bit)) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
  if (e == hipSuccess && d < 64) devices.fetch_or(bit, std::memory_order_relaxed);
  return e;
}

}  // namespace s2
