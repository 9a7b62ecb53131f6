// What launches share (host code).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

// Lets a kernel have ``bytes`` of dynamic LDS, once on every device and from any thread.  What fails
// here fails again as the launch's own error, which the caller asks for.
template <auto KERNEL>
static void allow_lds(int bytes) {
  static std::atomic<uint64_t> allowed{0};  // a bit a device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return;
  const uint64_t bit = 1ull << (device & 63);
  if (allowed.load(std::memory_order_acquire) & bit) return;
  if (hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) ==
      hipSuccess)
    allowed.fetch_or(bit, std::memory_order_release);
}
