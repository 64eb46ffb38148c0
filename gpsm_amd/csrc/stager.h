// Copies between ordinary host memory and the device, staged through pinned
// buffers of the context by several host threads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace gpsm {

// memcpy by up to eight threads (host/copy.cpp).
void parallel_copy(void* dst, const void* src, size_t n);

// The runtime stages a pageable copy itself, 1 MB at a time with one thread:
// about 60 us per MB to the device, and 130 us from it into memory that is
// touched for the first time, of which the copy engine takes 20 to 25.  Here
// the threads copy (and take the page faults of) one half of the staging while
// the other moves.  The edge list and CSR of a 1M-vertex graph (137 MB) took
// 9 of the 13.4 ms of building it.
//
// Used by the thread that uses the context, on its stream; copies of less
// than kMin bytes, or without memory for the staging, are the runtime's.
class Stager {
 public:
  static constexpr size_t kChunk = 4u << 20, kMin = 1u << 20;

  // src has been read on return; the copy to dst is queued on s.
  hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t s);
  // dst holds the data on return (everything before on s is waited for).
  hipError_t to_host(void* dst, const void* src, size_t n, hipStream_t s);
  void release();

 private:
  bool ready();
  char* half_[2] = {nullptr, nullptr};
  hipEvent_t moved_[2] = {nullptr, nullptr};  // the half's last copy
};

}  // namespace gpsm
