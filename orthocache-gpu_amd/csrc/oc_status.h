#pragma once
// Helpers shared by the C-ABI translation units: fail() records a message
// for oc_last_error() (thread-local) and returns the status code; device_cus().
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>

#include "orthocache_hip.h"

namespace oc {

void set_last_error(const char* msg);

__attribute__((format(printf, 2, 3))) inline int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  set_last_error(buf);
  return code;
}

inline int hip_fail(hipError_t e, const char* what) {
  return fail(OC_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

// CU count of the current device, cached per device index (a query costs
// about 0.3 us, and a launch's rules ask several times).
inline int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (!n) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace oc
