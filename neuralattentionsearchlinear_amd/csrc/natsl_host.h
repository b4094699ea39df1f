// Host-side helpers shared by the C-ABI entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <atomic>

#include "../../include/natsl.h"

namespace natsl {

char* error_buffer();  // thread-local, 512 bytes (defined in natsl_route.hip)

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(error_buffer(), 512, fmt, ap);
  va_end(ap);
  return code;
}

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
  return NATSL_OK;
}

// The LDS reservation of a kernel is an attribute of the function per device: set when a device first runs it.
inline int reserve_lds(const void* kern, std::atomic<unsigned long long>& done, size_t lds, const char* what) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: cannot name the current device (%s)", what, hipGetErrorString(e));
  const unsigned long long bit = 1ull << (dev & 63);
  if (dev < 64 && (done.load(std::memory_order_acquire) & bit)) return NATSL_OK;
  e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS: %s", what, lds, hipGetErrorString(e));
  if (dev < 64) done.fetch_or(bit, std::memory_order_release);
  return NATSL_OK;
}

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

}  // namespace natsl
