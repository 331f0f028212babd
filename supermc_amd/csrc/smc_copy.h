// smc_copy.h -- device-to-host copies into ordinary (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace smc {

// Copies of at least kStagedBytes into pageable memory go through pinned
// slots, one per worker thread: each worker takes the next kSlotBytes piece,
// queues its transfer into its slot and moves it on to the destination while
// the other workers' transfers run.  One thread through the runtime's own
// staging reaches 10 GB/s on untouched pages (17 on touched ones); a
// transfer into pinned memory runs at 57 GB/s and eight threads write 67 GB/s
// to untouched pages.  Smaller copies, pinned destinations, a stream of
// another device than the thread's, and copies for which no slot can be had
// take one hipMemcpyAsync; with some of the slots there are fewer workers.
//
// One object per context or handle; not thread-safe, like them.  The slots
// (at most kWorkers of them) are allocated by the first staged copy and freed
// with the object.
class HostCopier {
 public:
  static constexpr int kWorkers = 8;
  static constexpr size_t kSlotBytes = (size_t)2 << 20;
  static constexpr size_t kStagedBytes = (size_t)4 << 20;

  HostCopier() = default;
  HostCopier(const HostCopier&) = delete;
  HostCopier& operator=(const HostCopier&) = delete;
  ~HostCopier();

  // bytes from device memory src to host memory dst, after the work queued
  // on stream.  The destination is complete when the call has returned and
  // the stream has been waited for (a staged copy is complete on return).
  hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t stream);

  // whether copy() would stage these bytes
  static bool staged(const void* dst, size_t bytes);

 private:
  bool reserve(int i);
  void* slot_[kWorkers] = {};
  hipEvent_t done_[kWorkers] = {};
};

// memcpy by several threads where that pays
void parallel_memcpy(void* dst, const void* src, size_t bytes);

}  // namespace smc
