// smc_copy.cpp -- pageable device-to-host copies by worker threads (smc_copy.h)
#include "smc_copy.h"

#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

namespace smc {

namespace {

int workers_for(size_t pieces) {
  const int hc = (int)std::thread::hardware_concurrency();
  return (int)std::min<size_t>(pieces, (size_t)std::max(1, std::min(HostCopier::kWorkers, hc / 2)));
}

// f(0) .. f(n - 1) at once, n <= kWorkers, f(0) on this thread; where a thread
// cannot be started (no thread, no memory), on this one
template <class F>
void run_workers(int n, const F& f) noexcept {
  std::thread th[HostCopier::kWorkers];
  for (int i = 1; i < n; ++i) {
    try {
      th[i] = std::thread(f, i);
    } catch (...) {
    }
  }
  f(0);
  for (int i = 1; i < n; ++i)
    if (!th[i].joinable()) f(i);
  for (int i = 1; i < n; ++i)
    if (th[i].joinable()) th[i].join();
}

}  // namespace

HostCopier::~HostCopier() {
  for (hipEvent_t e : done_)
    if (e) (void)hipEventDestroy(e);
  if (slots_) (void)hipHostFree(slots_);
}

// whether most pages of the destination have not been touched yet (four are
// looked at)
static bool untouched(const void* dst, size_t bytes) {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE);
  int fresh = 0;
  for (int i = 0; i < 4; ++i) {
    const uintptr_t at = ((uintptr_t)dst + bytes / 8 * (2 * i + 1)) / page * page;
    unsigned char in_memory = 1;
    if (mincore((void*)at, page, &in_memory) == 0 && !(in_memory & 1)) ++fresh;
  }
  return fresh > 2;
}

// How many of n workers have a slot and an event for a copy of these bytes;
// where they cannot be had, no error is left behind.
int HostCopier::reserve(int n, const void* dst, size_t bytes) {
  if (!slots_) {
    saved_us_ += (double)bytes / (1 << 20) * (untouched(dst, bytes) ? kFreshUs : kWrittenUs);
    if (saved_us_ < kSlotsUs) return 0;
    saved_us_ = 0;
    if (hipHostMalloc((void**)&slots_, kWorkers * kSlotBytes, hipHostMallocDefault) != hipSuccess) {
      slots_ = nullptr;
      (void)hipGetLastError();
      return 0;
    }
  }
  for (int i = 0; i < n; ++i)
    if (!done_[i] && hipEventCreateWithFlags(&done_[i], hipEventDisableTiming) != hipSuccess) {
      done_[i] = nullptr;
      (void)hipGetLastError();
      return i;
    }
  return n;
}

bool HostCopier::staged(const void* dst, size_t bytes) {
  if (bytes < kStagedBytes) return false;
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, dst) != hipSuccess) {
    (void)hipGetLastError();  // memory the runtime does not know: pageable
    return true;
  }
  return at.type == hipMemoryTypeUnregistered;
}

hipError_t HostCopier::copy(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  const size_t pieces = (bytes + kSlotBytes - 1) / kSlotBytes;
  int n = 0, dev = 0, of_stream = -1;  // n workers have a slot and an event
  if (staged(dst, bytes)) {
    if (hipGetDevice(&dev) == hipSuccess && hipStreamGetDevice(stream, &of_stream) == hipSuccess) {
      if (of_stream == dev) n = reserve(workers_for(pieces), dst, bytes);
    } else {
      (void)hipGetLastError();
    }
  }
  if (n == 0) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  std::mutex order;  // pieces are queued in the order they are taken
  const auto work = [&](int i) {
    if (i > 0 && hipSetDevice(dev) != hipSuccess) return;  // the pieces are left to the others
    char* const slot = slots_ + (size_t)i * kSlotBytes;
    while (err.load() == (int)hipSuccess) {
      size_t off, m;
      hipError_t e;
      {
        const std::lock_guard<std::mutex> g(order);
        const size_t p = next++;
        if (p >= pieces) return;
        off = p * kSlotBytes;
        m = std::min(kSlotBytes, bytes - off);
        e = hipMemcpyAsync(slot, (const char*)src + off, m, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(done_[i], stream);
      }
      if (e == hipSuccess) e = hipEventSynchronize(done_[i]);
      if (e != hipSuccess) {
        err = (int)e;
        return;
      }
      std::memcpy((char*)dst + off, slot, m);
    }
  };
  run_workers(n, work);
  return (hipError_t)err.load();
}

void parallel_memcpy(void* dst, const void* src, size_t bytes) {
  constexpr size_t kPiece = (size_t)1 << 20;
  const int n = bytes < (size_t)4 << 20 ? 1 : workers_for(bytes / kPiece);
  const size_t per = ((bytes + n - 1) / n + 4095) & ~(size_t)4095;  // n pieces of whole pages cover all bytes
  run_workers(n, [&](int i) {
    const size_t off = std::min(bytes, per * i), m = std::min(per, bytes - off);
    if (m) std::memcpy((char*)dst + off, (const char*)src + off, m);
  });
}

}  // namespace smc
