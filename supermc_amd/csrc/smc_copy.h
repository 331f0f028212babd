// smc_copy.h -- device-to-host copies into ordinary (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace smc {

// Copies of at least kStagedBytes into pageable memory go through pinned
// slots (once there are slots, below), one per worker thread: each worker takes the next kSlotBytes piece,
// queues its transfer into its slot and moves it on to the destination while
// the other workers' transfers run.  One thread through the runtime's own
// staging reaches 10 GB/s on untouched pages (17 on touched ones); a
// transfer into pinned memory runs at 57 GB/s and eight threads write 67 GB/s
// to untouched pages.  Smaller copies, pinned destinations, a stream of
// another device than the thread's, and copies for which no slot can be had
// take one hipMemcpyAsync.
//
// One object per context or handle; not thread-safe, like them.  The slots
// (one block for kWorkers of them, freed with the object) take 1.4 ms to make,
// and a copy through them saves 185 us per MiB of a destination whose pages
// are untouched and 32 us of one already written: they are made for the copy
// with which the object's copies would have saved as much.  Made for the first
// 4 MiB, they had the first 20 FP64 grids of a context (11 MB, written before)
// take 2.4 ms instead of 1.7.
class HostCopier {
 public:
  static constexpr int kWorkers = 8;
  static constexpr size_t kSlotBytes = (size_t)2 << 20;
  static constexpr size_t kStagedBytes = (size_t)4 << 20;
  static constexpr double kSlotsUs = 1400, kFreshUs = 185, kWrittenUs = 32;  // to make the slots; saved per MiB

  HostCopier() = default;
  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;
  ~HostCopier();

  // bytes from device memory src to host memory dst, after the work queued
  // on stream.  The destination is complete when the call has returned and
  // the stream has been waited for (a staged copy is complete on return).
  hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t stream);

  // whether these bytes are worth staging, given the slots
  static bool staged(const void* dst, size_t bytes);

 private:
  int reserve(int n, const void* dst, size_t bytes);
  char* slots_ = nullptr;
  hipEvent_t done_[kWorkers] = {};
  double saved_us_ = 0;  // what slots would have saved, until there are some
};

// memcpy by several threads where that pays
void parallel_memcpy(void* dst, const void* src, size_t bytes);

}  // namespace smc
