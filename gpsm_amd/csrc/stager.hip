// Stager (stager.h).
#include "stager.h"

#include <algorithm>

namespace gpsm {

bool Stager::ready() {
  for (int i = 0; i < 2; ++i) {
    if (!half_[i]) {
      void* p = nullptr;
      if (hipHostMalloc(&p, kChunk, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      half_[i] = static_cast<char*>(p);
    }
    if (!moved_[i] && hipEventCreateWithFlags(&moved_[i], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      moved_[i] = nullptr;
      return false;
    }
  }
  return true;
}

void Stager::release() {
  for (int i = 0; i < 2; ++i) {
    if (half_[i]) hipHostFree(half_[i]);
    if (moved_[i]) hipEventDestroy(moved_[i]);
    half_[i] = nullptr;
    moved_[i] = nullptr;
  }
}

hipError_t Stager::to_device(void* dst, const void* src, size_t n, hipStream_t s) {
  if (!n) return hipSuccess;
  if (n < kMin || !ready()) return hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s);
  int i = 0;
  for (size_t at = 0; at < n; at += kChunk, i ^= 1) {
    const size_t m = std::min(kChunk, n - at);
    hipError_t e = hipEventSynchronize(moved_[i]);  // an event never recorded is complete
    if (e != hipSuccess) return e;
    parallel_copy(half_[i], static_cast<const char*>(src) + at, m);
    if ((e = hipMemcpyAsync(static_cast<char*>(dst) + at, half_[i], m, hipMemcpyHostToDevice, s)) != hipSuccess ||
        (e = hipEventRecord(moved_[i], s)) != hipSuccess)
      return e;
  }
  return hipSuccess;
}

hipError_t Stager::to_host(void* dst, const void* src, size_t n, hipStream_t s) {
  if (!n) return hipStreamSynchronize(s);
  if (n < kMin || !ready()) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);
    return e != hipSuccess ? e : w;
  }
  const size_t chunks = (n + kChunk - 1) / kChunk;
  for (size_t k = 0; k <= chunks; ++k) {
    // chunk k moves while chunk k - 1 is copied out; on one stream the copies
    // that still read a half from to_device are done before it is written
    if (k < chunks) {
      const size_t at = k * kChunk, m = std::min(kChunk, n - at);
      hipError_t e;
      if ((e = hipMemcpyAsync(half_[k & 1], static_cast<const char*>(src) + at, m, hipMemcpyDeviceToHost, s)) !=
              hipSuccess ||
          (e = hipEventRecord(moved_[k & 1], s)) != hipSuccess) {
        (void)hipStreamSynchronize(s);
        return e;
      }
    }
    if (k > 0) {
      const size_t at = (k - 1) * kChunk;
      const hipError_t e = hipEventSynchronize(moved_[(k - 1) & 1]);
      if (e != hipSuccess) return e;
      parallel_copy(static_cast<char*>(dst) + at, half_[(k - 1) & 1], std::min(kChunk, n - at));
    }
  }
  return hipSuccess;
}

}  // namespace gpsm
