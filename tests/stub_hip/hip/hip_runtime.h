// The few HIP calls that the block pool makes, over a device of a fixed size:
// the pool's logic on the CPU.
#pragma once
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };

namespace stub {
inline std::mutex lock;
inline std::map<uintptr_t, size_t> live;
inline size_t room = 0, bad_frees = 0;  // bytes left; frees of what is not allocated
inline uintptr_t next = 4096;
}  // namespace stub

template <typename T>
inline hipError_t hipMalloc(T** p, size_t n) {
  std::lock_guard<std::mutex> l(stub::lock);
  if (n > stub::room) return hipErrorOutOfMemory;
  stub::room -= n;
  stub::live[stub::next] = n;
  *p = reinterpret_cast<T*>(stub::next);
  stub::next += n + 4096;
  return hipSuccess;
}

inline hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(stub::lock);
  auto it = stub::live.find(reinterpret_cast<uintptr_t>(p));
  if (it == stub::live.end()) {
    ++stub::bad_frees;
    return hipSuccess;
  }
  stub::room += it->second;
  stub::live.erase(it);
  return hipSuccess;
}

inline hipError_t hipGetLastError() { return hipSuccess; }
