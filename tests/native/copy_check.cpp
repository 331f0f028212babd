// copy_check.cpp -- smc_copy.cpp on the CPU: the check named on the command
// line, 0 if it holds.  The HIP calls it makes are defined here, over host
// memory: transfers are done when they are queued.
#include <sys/mman.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "../../supermc_amd/csrc/smc_copy.h"

// allocations left before one fails (negative: none fails)
static thread_local int g_allocations = -1;

void* operator new(size_t n) {
  if (g_allocations >= 0 && g_allocations-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// calls left before the kind fails from then on (negative: it does not fail)
static int g_slots = -1, g_events = -1, g_device = -1, g_threads = -1;
static hipError_t g_last = hipSuccess;
static int g_stream_device = 0, g_made = 0;

static hipError_t after(int& left, hipError_t e) {
  if (left < 0 || left-- > 0) return hipSuccess;
  left = 0;
  return g_last = e;
}

extern "C" {
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return after(g_device, hipErrorNoDevice);
}
hipError_t hipSetDevice(int) {
  static std::mutex one;
  const std::lock_guard<std::mutex> g(one);
  return after(g_threads, hipErrorInvalidDevice);
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* d) {
  *d = g_stream_device;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++g_made;
  const hipError_t e = after(g_slots, hipErrorOutOfMemory);
  if (e == hipSuccess) *p = std::malloc(n);
  return e;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* p, unsigned) {
  const hipError_t e = after(g_events, hipErrorOutOfMemory);
  if (e == hipSuccess) *p = (hipEvent_t)std::malloc(1);
  return e;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void*)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  return g_stream_device == 0 ? hipSuccess : hipErrorInvalidHandle;  // events are of device 0
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
}

namespace {

int fail(const char* what, size_t at) {
  std::fprintf(stderr, "%s (%zu)\n", what, at);
  return 1;
}

std::vector<unsigned char> pattern(size_t n) {
  std::vector<unsigned char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (unsigned char)(1 + i % 251);
  return v;
}

// every byte arrives, none past the end is written: counts around whole
// pages per worker for any number of workers, and the smallest
int check_memcpy() {
  const auto src = pattern((size_t)17 << 20);
  std::vector<unsigned char> dst(src.size());
  for (size_t mib : {0, 4, 5, 6, 7, 8, 12, 16})
    for (int r = mib ? -9 : 0; r <= 9; ++r) {
      const size_t n = (mib << 20) + r;
      std::fill(dst.begin(), dst.begin() + n + 64, 0);
      smc::parallel_memcpy(dst.data(), src.data(), n);
      if (std::memcmp(dst.data(), src.data(), n) != 0) return fail("bytes missing", n);
      for (size_t i = n; i < n + 64; ++i)
        if (dst[i]) return fail("written past the end", n);
    }
  return 0;
}

// the bytes arrive, and no exception leaves the call, when any one of its
// allocations (a thread's state) fails
int check_allocations() {
  const auto src = pattern((size_t)8 << 20);
  std::vector<unsigned char> dst(src.size());
  for (int k = 0; k < 2 * smc::HostCopier::kWorkers; ++k) {
    std::fill(dst.begin(), dst.end(), 0);
    try {
      g_allocations = k;
      smc::parallel_memcpy(dst.data(), src.data(), src.size());
    } catch (...) {
      return fail("exception", k);
    }
    g_allocations = -1;
    if (dst != src) return fail("bytes missing", k);
  }
  return 0;
}

// a large copy succeeds and leaves no error behind when the k-th and every
// later slot, event, device query or worker's device call fails
int check_slots() {
  const auto src = pattern(((size_t)45 << 20) + 5);
  std::vector<unsigned char> dst(src.size());
  for (int* left : {&g_slots, &g_events, &g_device, &g_threads})
    for (int k = 0; k < smc::HostCopier::kWorkers; ++k) {
      smc::HostCopier copier;
      for (int again = 0; again < 2; ++again) {  // the second call after the first could not get everything
        std::fill(dst.begin(), dst.end(), 0);
        *left = k;
        const hipError_t e = copier.copy(dst.data(), src.data(), src.size(), nullptr);
        *left = -1;
        if (e != hipSuccess) return fail("error returned", k);
        if (dst != src) return fail("bytes missing", k);
        if (left != &g_threads && hipGetLastError() != hipSuccess) return fail("error left behind", k);
      }
    }
  smc::HostCopier copier;
  g_stream_device = 1;
  std::fill(dst.begin(), dst.end(), 0);
  if (copier.copy(dst.data(), src.data(), src.size(), nullptr) != hipSuccess || dst != src)
    return fail("stream of another device", 1);
  return 0;
}

// Slots are made once, for the copy with which the copies so far would have
// saved the time: after 44 MiB into written pages, 8 MiB into untouched ones.
int check_first() {
  const auto src = pattern((size_t)16 << 20);
  for (const bool fresh : {false, true})
    for (size_t mib : {3, 4, 5, 6, 8, 15, 16}) {
      smc::HostCopier copier;
      g_made = 0;
      double saved = 0;
      for (int k = 0; k < 12; ++k) {
        const size_t n = mib << 20;
        char* dst = (char*)mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (!fresh) std::memset(dst, 1, n);
        if (copier.copy(dst, src.data(), n, nullptr) != hipSuccess || std::memcmp(dst, src.data(), n) != 0)
          return fail("bytes missing", mib);
        munmap(dst, n);
        if (n >= smc::HostCopier::kStagedBytes)
          saved += (double)mib * (fresh ? smc::HostCopier::kFreshUs : smc::HostCopier::kWrittenUs);
        if (g_made != (saved >= smc::HostCopier::kSlotsUs ? 1 : 0)) return fail("slots made", mib);
      }
    }
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const char* name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "memcpy")) return check_memcpy();
  if (!std::strcmp(name, "allocations")) return check_allocations();
  if (!std::strcmp(name, "slots")) return check_slots();
  if (!std::strcmp(name, "first")) return check_first();
  return fail("no such check", 0);
}
