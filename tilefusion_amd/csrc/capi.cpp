// Error reporting and version of the C ABI (declared in include/tilefusion_c.h).
#include <atomic>
#include <chrono>
#include <cstring>

#include "common.hpp"

namespace tfk {
namespace {
thread_local char g_last_error[4096] = "";  // room for a compiler diagnostic
}

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
}

int hip_fail(hipError_t e, const char* what) {
  set_error("HIP error '%s' from %s", hipGetErrorString(e), what);
  return TF_ERR_HIP;
}

bool is_ordinary_device_memory(const void* p) {
  int device = -1;
  hipPointerAttribute_t a{};
  if (hipGetDevice(&device) != hipSuccess || hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();   // not an error of this call
    return false;
  }
  return a.type == hipMemoryTypeDevice && !a.isManaged && a.device == device && a.allocationFlags == hipDeviceMallocDefault;
}

arrivals_t next_arrivals_tag() {
  // splitmix64 over a count that starts differently in every process, 48 bits of it: tags look like nothing that a workspace holds (counts or
  // addresses might).  Two launches may have the same one (to be expected within some 2^24 of them); nothing rests on it, as no launch
  // leaves its tag behind.
  static std::atomic<unsigned long long> count{
      (unsigned long long)std::chrono::system_clock::now().time_since_epoch().count() ^ (unsigned long long)(uintptr_t)&count};
  for (;;) {
    unsigned long long x = count.fetch_add(0x9e3779b97f4a7c15ull, std::memory_order_relaxed);
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    x = (x ^ (x >> 31)) & ~kArrivalsMask;
    if (x != 0) return x;   // (zero is what a word without arrivals holds)
  }
}
}  // namespace tfk

extern "C" {
const char* tf_last_error(void) { return tfk::g_last_error; }
const char* tf_version(void) { return "tilefusion-mi355x 0.1.0 (gfx950)"; }
}
