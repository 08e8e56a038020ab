// hostcopy.h -- large copies between device memory and a caller's pageable array.
#pragma once
#include <cstddef>

#include <hip/hip_runtime.h>

namespace mgd {

// Pinned staging of one region's large state copies, allocated at the first one and given back
// with the region.  One copy at a time (a region's entry points are not called concurrently).
class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy();
  // Copies `bytes` on `st`, after the work enqueued there, and returns when the data is there.
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t st);

 private:
  static constexpr size_t kChunk = size_t(2) << 20;
  static constexpr int kMostSlots = 16;
  bool prepare(int slots, hipStream_t st);
  bool make(int slots);
  char* buf_ = nullptr;
  int slots_ = 0;
  hipEvent_t ev_[kMostSlots] = {};
  bool failed_ = false;
};

}  // namespace mgd
