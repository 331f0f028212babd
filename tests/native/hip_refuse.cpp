// hip_refuse.cpp -- a hipMalloc that refuses allocations from a size on, for
// tests of what is done without the memory.  Loaded with RTLD_GLOBAL before
// the libraries that call hipMalloc.
#include <hip/hip_runtime_api.h>

static hipError_t (*g_real)(void**, size_t) = nullptr;
static size_t g_from = ~(size_t)0;
static int g_refused = 0;

extern "C" {
void refuse_init(void* real) { g_real = (hipError_t(*)(void**, size_t))real; }
void refuse_from(size_t bytes) { g_from = bytes; }
int refuse_count() { return g_refused; }

hipError_t hipMalloc(void** p, size_t n) {
  if (n >= g_from) {
    ++g_refused;
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  return g_real(p, n);
}
}
