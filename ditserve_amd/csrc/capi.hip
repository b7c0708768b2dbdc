// C-ABI plumbing: per-thread error message, version, launch checks.
#include <stdarg.h>
#include <stdio.h>

#include <atomic>

#include "ditk_common.h"

namespace {
thread_local char g_err[512] = "";
}

void ditk_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int ditk_check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    ditk_set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return 2;
  }
  return 0;
}

// Cached per device (callers on several host threads may race to fill an entry; they
// store the same value).
int ditk_cu_count() {
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int c = cached[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    int n = 0;
    c = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    cached[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

DITK_EXPORT const char* ditk_last_error(void) { return g_err; }

DITK_EXPORT int ditk_version(void) { return 1; }
