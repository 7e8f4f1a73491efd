// Workspaces of extended shapes on a device whose memory ends at a limit
// (linked with --wrap for the three calls below, so it needs no device).
// Prints, per line of "limit held want enough", what the pool returned, holds
// and was asked for, or "error <code>".
#include <cstdio>
#include <cstdlib>

#include "conv_driver.hpp"

using namespace fcamd;

static size_t g_limit, g_last;

extern "C" hipError_t __wrap_hipMalloc(void** p, size_t bytes) {
  g_last = bytes;
  if (bytes > g_limit) return hipErrorOutOfMemory;
  *p = std::malloc(16);
  return hipSuccess;
}
extern "C" hipError_t __wrap_hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
extern "C" hipError_t __wrap_hipDeviceSynchronize() { return hipSuccess; }

int main() {
  size_t held, want, enough;
  while (std::scanf("%zu %zu %zu %zu", &g_limit, &held, &want, &enough) == 4) {
    DevicePool pool;
    g_last = 0;
    if (held) {
      pool.ws = std::malloc(16);
      pool.ws_bytes = held;
    }
    try {
      const size_t got = pool_reserve_workspace(pool, want, enough);
      std::printf("%zu %zu %zu\n", got, pool.ws ? pool.ws_bytes : 0, g_last);
    } catch (const Error& e) {
      std::printf("error %d %zu\n", e.code, pool.ws ? pool.ws_bytes : (size_t)0);
    }
    std::free(pool.ws);
  }
  return 0;
}
