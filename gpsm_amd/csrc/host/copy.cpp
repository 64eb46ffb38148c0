// Large host copies by several threads: one thread's memcpy reaches a quarter
// of the copy engine's rate, less into pages touched for the first time.
#include <omp.h>

#include <algorithm>
#include <cstddef>
#include <cstring>

namespace gpsm {

void parallel_copy(void* dst, const void* src, size_t n) {
  constexpr size_t kPart = 256u << 10;  // bytes worth a thread
  const int threads = (int)std::min<size_t>({8, (size_t)std::max(omp_get_max_threads(), 1), n / kPart});
  if (threads < 2) {
    std::memcpy(dst, src, n);
    return;
  }
#pragma omp parallel num_threads(threads)
  {
    // pages are not shared between threads
    const size_t t = (size_t)omp_get_thread_num(), k = (size_t)omp_get_num_threads();
    const size_t page = 4096, pages = (n + page - 1) / page;
    const size_t lo = std::min(n, pages * t / k * page), hi = std::min(n, pages * (t + 1) / k * page);
    if (hi > lo) std::memcpy(static_cast<char*>(dst) + lo, static_cast<const char*>(src) + lo, hi - lo);
  }
}

}  // namespace gpsm
