// What calls leave for the next call (host code, no HIP types: the library and
// the CPU checks share it).
#pragma once

#include <cstddef>
#include <list>
#include <memory>
#include <mutex>
#include <utility>

namespace ccpi {

// Idle objects of type T (T::bytes() of memory each) by device, lent to one
// holder at a time.  At most `count` of them and `bytes` of memory together
// stay: the ones left last do, and one of more than `bytes` never.  Objects
// that do not stay are destroyed outside the lock (freeing device memory
// waits for the device).
template <class T>
class Kept {
 public:
  Kept(size_t count, size_t bytes) : count_(count), bytes_(bytes) {}

  // The one left last on `dev`, or none.
  std::unique_ptr<T> take(int dev) {
    std::lock_guard<std::mutex> lk(mu_);
    for (auto it = idle_.begin(); it != idle_.end(); ++it)
      if (it->first == dev) {
        std::unique_ptr<T> t = std::move(it->second);
        idle_.erase(it);
        return t;
      }
    return nullptr;
  }

  void leave(int dev, std::unique_ptr<T> t) noexcept {
    if (t->bytes() > bytes_) return;
    List over;
    try {
      List one;
      one.emplace_front(dev, std::move(t));
      std::lock_guard<std::mutex> lk(mu_);
      idle_.splice(idle_.begin(), one);
      size_t n = 0, b = 0;
      for (auto it = idle_.begin(); it != idle_.end();) {
        const auto q = it++;
        n++;
        b += q->second->bytes();
        if (n > count_ || b > bytes_) {
          b -= q->second->bytes();
          n--;
          over.splice(over.end(), idle_, q);
        }
      }
    } catch (...) {
      // no host memory for the list: not kept
    }
  }

  // Destroys the idle ones.
  void give_back() {
    List all;
    std::lock_guard<std::mutex> lk(mu_);
    all.swap(idle_);
  }

 private:
  using List = std::list<std::pair<int, std::unique_ptr<T>>>;
  const size_t count_, bytes_;
  std::mutex mu_;
  List idle_;   // last left first
};

// alloc()'s status; where it is `refused`, that of a second try after
// give_back().
template <class Status, class Alloc, class GiveBack>
Status alloc_giving_back(Status refused, Alloc &&alloc, GiveBack &&give_back) {
  Status s = alloc();
  if (s == refused) {
    give_back();
    s = alloc();
  }
  return s;
}

}  // namespace ccpi
