// The block pool over a device of fixed size (stub_hip): prints one line per
// check that fails, "ok" at the end.
#include <atomic>
#include <cstdio>
#include <set>
#include <thread>

#include "pool.h"

using gpsm::BlockPool;
using gpsm::device_malloc;

#define CHECK(x) \
  if (!(x)) std::printf("failed: %s (line %d)\n", #x, __LINE__)

constexpr size_t MB = 1u << 20;

// An allocation outside the pools, or of another context's pool, gets what waits in one.
void idle_memory_goes_back() {
  stub::room = 100 * MB;
  BlockPool a, b;
  void* p = a.take(80 * MB);
  CHECK(p && stub::room == 20 * MB);
  a.give(p);
  CHECK(stub::room == 20 * MB);
  char* x = nullptr;
  CHECK(device_malloc(&x, 50 * MB) && x && stub::room == 50 * MB);
  hipFree(x);
  p = a.take(80 * MB);
  a.give(p);
  void* q = b.take(90 * MB);
  CHECK(q && stub::room == 10 * MB);
  CHECK(!a.take(20 * MB));
  CHECK(!device_malloc(&x, 20 * MB) && !x);
  b.give(q);
  CHECK(b.take(90 * MB) == q);  // reused, not allocated
  b.give(q);
  a.release();
  b.release();
  CHECK(stub::room == 100 * MB && stub::live.empty());
}

// Blocks taken, given back and released by several threads at once.
void threads() {
  stub::room = 64 * MB;
  BlockPool pool;
  std::mutex lock;
  std::set<void*> held;
  std::atomic<int> doubles{0};
  auto work = [&](int t) {
    for (int i = 0; i < 20000; ++i) {
      void* p = pool.take((1 + (t + i) % 7) * 100000);
      if (!p) continue;
      {
        std::lock_guard<std::mutex> l(lock);
        if (!held.insert(p).second) ++doubles;
      }
      if (i % 512 == t) {
        char* x = nullptr;  // sometimes finds no memory and empties the pool
        if (device_malloc(&x, 60 * MB)) hipFree(x);
      }
      {
        std::lock_guard<std::mutex> l(lock);
        held.erase(p);
      }
      pool.give(p);
    }
  };
  std::thread ts[4];
  for (int t = 0; t < 4; ++t) ts[t] = std::thread(work, t);
  for (auto& t : ts) t.join();
  pool.release();
  CHECK(doubles == 0 && stub::bad_frees == 0);
  CHECK(stub::live.empty() && stub::room == 64 * MB);
}

int main() {
  idle_memory_goes_back();
  threads();
  std::printf("ok\n");
}
