// Library-level entry points: version string, per-thread error messages and
// the device's size.
#include "common.h"

#include <atomic>

namespace cs {
namespace {
thread_local char g_error[512] = "";
}

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int compute_units() {
  static std::atomic<int> cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}
}  // namespace cs

extern "C" const char* cs_version(void) { return "cacheslide_hip 0.1.0 gfx950"; }

extern "C" const char* cs_last_error(void) { return cs::g_error; }
