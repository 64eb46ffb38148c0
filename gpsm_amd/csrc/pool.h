// Device memory of resident graphs and of building them, reused by a
// context's later graphs.
//
// A graph of 1M vertices takes 3.2 GB (hub bitmaps) and 0.5 GB while it is
// built.  Returned to the driver at once, such blocks cost more than the
// build: after about 45 graphs made and freed one after the other every
// hipFree of the bitmaps took 100 ms (17 ms per graph before, 121 ms after;
// 43 ms with the slower host build, which the driver kept up with).
//
// One pool per context, used by the thread that uses the context; a block is
// handed out again only to work on the context's stream, which its last user
// waited for.  At most kMost bytes wait for reuse; they go back when the
// context ends or when one of its allocations fails.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <unordered_map>
#include <vector>

namespace gpsm {

class BlockPool {
 public:
  static constexpr size_t kMost = 8ull << 30;

  // At least nbytes (nullptr: no memory).
  void* take(size_t nbytes) {
    nbytes = nbytes ? (nbytes + 255) & ~(size_t)255 : 256;
    size_t best = idle_.size();
    for (size_t i = 0; i < idle_.size(); ++i)
      if (idle_[i].bytes >= nbytes && idle_[i].bytes <= nbytes + nbytes / 8 &&
          (best == idle_.size() || idle_[i].bytes < idle_[best].bytes))
        best = i;
    Block b{nullptr, nbytes};
    if (best < idle_.size()) {
      b = idle_[best];
      idle_.erase(idle_.begin() + best);
      waiting_ -= b.bytes;
    } else if (hipMalloc(&b.ptr, nbytes) != hipSuccess) {
      (void)hipGetLastError();
      release();
      if (hipMalloc(&b.ptr, nbytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
      }
    }
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
    for (auto& b : idle_) hipFree(b.ptr);
    idle_.clear();
    waiting_ = 0;
  }

 private:
  struct Block {
    void* ptr;
    size_t bytes;
  };
  std::vector<Block> idle_;
  size_t waiting_ = 0;
  std::unordered_map<void*, size_t> used_;
};

}  // namespace gpsm
