// Device memory of resident graphs and of building them, reused by a
// context's later graphs.
//
// A graph of 1M vertices takes 3.2 GB (hub bitmaps) and 0.5 GB while it is
// built.  Returned to the driver at once, such blocks cost more than the
// build: after about 45 graphs made and freed one after the other every
// hipFree of the bitmaps took 100 ms (17 ms per graph before, 121 ms after;
// 43 ms with the slower host build, which the driver kept up with).
//
// One pool per context; a block is handed out again only to work on the
// context's stream, which its last user waited for.  A graph may be freed by
// another thread than the context's (a Python reference dropped there), so a
// lock guards the pool.  At most kMost bytes wait for reuse; they go back when
// the context ends or when any allocation of the library fails, on whichever
// thread and of whichever context (device_malloc).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace gpsm {

class BlockPool {
 public:
  static constexpr size_t kMost = 8ull << 30;

  BlockPool() {
    std::lock_guard<std::mutex> l(all().lock);
    all().pools.push_back(this);
  }
  ~BlockPool() {
    std::lock_guard<std::mutex> l(all().lock);
    auto& v = all().pools;
    v.erase(std::find(v.begin(), v.end(), this));
  }
  BlockPool(const BlockPool&) = delete;
  BlockPool& operator=(const BlockPool&) = delete;

  // At least nbytes (nullptr: no memory).
  void* take(size_t nbytes) {
    nbytes = nbytes ? (nbytes + 255) & ~(size_t)255 : 256;
    Block b = idle_block(nbytes);
    // not under the lock: a failed allocation empties every pool, this one too
    if (!b.ptr && !allocate(&b.ptr, nbytes)) return nullptr;
    std::lock_guard<std::mutex> l(lock_);
    used_[b.ptr] = b.bytes;
    return b.ptr;
  }

  template <typename T>
  bool take(T** p, size_t count) {
    return (*p = static_cast<T*>(take(sizeof(T) * count))) != nullptr;
  }

  // The block's last user has been waited for.
  void give(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> l(lock_);
    auto it = used_.find(p);
    if (it == used_.end()) return;
    const size_t bytes = it->second;
    used_.erase(it);
    if (bytes > kMost) {
      hipFree(p);
      return;
    }
    // the oldest leave first
    while (waiting_ + bytes > kMost) {
      hipFree(idle_.front().ptr);
      waiting_ -= idle_.front().bytes;
      idle_.erase(idle_.begin());
    }
    idle_.push_back({p, bytes});
    waiting_ += bytes;
  }

  // Everything that waits, back to the driver.
  void release() {
    std::lock_guard<std::mutex> l(lock_);
    for (auto& b : idle_) hipFree(b.ptr);
    idle_.clear();
    waiting_ = 0;
  }

  // hipMalloc, a second time without what waits in the pools.
  static bool allocate(void** p, size_t nbytes) {
    if (hipMalloc(p, nbytes) == hipSuccess) return true;
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> l(all().lock);
      for (BlockPool* x : all().pools) x->release();
    }
    if (hipMalloc(p, nbytes) == hipSuccess) return true;
    (void)hipGetLastError();
    *p = nullptr;
    return false;
  }

 private:
  struct Block {
    void* ptr;
    size_t bytes;
  };
  struct Pools {
    std::mutex lock;
    std::vector<BlockPool*> pools;
  };

  // The pools of all contexts; never destroyed, a context may end after main.
  static Pools& all() {
    static Pools* p = new Pools();
    return *p;
  }

  // The smallest block that waits and fits without much waste, taken out.
  Block idle_block(size_t nbytes) {
    std::lock_guard<std::mutex> l(lock_);
    size_t best = idle_.size();
    for (size_t i = 0; i < idle_.size(); ++i)
      if (idle_[i].bytes >= nbytes && idle_[i].bytes <= nbytes + nbytes / 8 &&
          (best == idle_.size() || idle_[i].bytes < idle_[best].bytes))
        best = i;
    if (best == idle_.size()) return {nullptr, nbytes};
    const Block b = idle_[best];
    idle_.erase(idle_.begin() + best);
    waiting_ -= b.bytes;
    return b;
  }

  std::mutex lock_;
  std::vector<Block> idle_;
  size_t waiting_ = 0;
  std::unordered_map<void*, size_t> used_;
};

// Device memory outside the pools; false (*p null) without memory.
template <typename T>
bool device_malloc(T** p, size_t nbytes) {
  return BlockPool::allocate(reinterpret_cast<void**>(p), nbytes);
}

}  // namespace gpsm
