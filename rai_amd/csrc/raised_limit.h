// A limit that calls raise as they need it, from any thread (no HIP here, so that
// the host can test it alone).
#ifndef RAI_RAISED_LIMIT_H
#define RAI_RAISED_LIMIT_H

#include <atomic>
#include <cstddef>
#include <mutex>

namespace rai {

// set(n) runs under the lock and only with a larger n than any before it, and
// raise(n) returns after a set of n or more: a caller that lost a race must
// neither lower the limit nor go on before it holds.
class RaisedLimit {
 public:
  template <class F>
  void raise(size_t n, F set) {
    if (n <= now_.load(std::memory_order_acquire)) return;
    std::lock_guard<std::mutex> lk(m_);
    if (n <= now_.load(std::memory_order_relaxed)) return;
    set(n);
    now_.store(n, std::memory_order_release);
  }

 private:
  std::mutex m_;
  std::atomic<size_t> now_{0};
};

}  // namespace rai

#endif
