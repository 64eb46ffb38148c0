// Objects kept for reuse, each lent to one caller at a time.
#pragma once
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

namespace gpsm {

// take() and give() may be called by several threads; as many objects exist
// as were ever lent out at the same time.
template <typename T>
class Leases {
 public:
  std::unique_ptr<T> take() {
    std::lock_guard<std::mutex> l(lock_);
    if (idle_.empty()) return std::make_unique<T>();
    std::unique_ptr<T> x = std::move(idle_.back());
    idle_.pop_back();
    return x;
  }

  void give(std::unique_ptr<T> x) {
    std::lock_guard<std::mutex> l(lock_);
    idle_.push_back(std::move(x));
  }

  // f(x) for every object that is not lent out.
  template <typename F>
  void each(F f) {
    std::lock_guard<std::mutex> l(lock_);
    for (auto& x : idle_) f(*x);
  }

 private:
  std::mutex lock_;
  std::vector<std::unique_ptr<T>> idle_;
};

}  // namespace gpsm
