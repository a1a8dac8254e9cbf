// Host buffers of the model calls: pageable memory to and from the device
// through pinned staging blocks and a few copy threads.
//
// hipMemcpyAsync on pageable memory moved 16.8 MB of hidden states at 12 to 15
// GB/s and took 30 to 70 us for a few kilobytes, each with a wait of its own
// (2.5 of the 6.5 ms of a 1024-token layer, half of a one-token layer).  Here a
// kernel reads or writes the pinned block directly (no copy engine hand-off),
// the host's copies run on several threads and overlap the device's piece by
// piece, and the call waits once.
#ifndef RAI_HOST_IO_H
#define RAI_HOST_IO_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace rai {

// Copies of 1 MB and more, in blocks that the caller and the pool's threads
// take in turn.  One copy at a time uses the threads; a second caller copies
// alone.  The threads sleep between copies and last as long as the process.
class CopyPool {
 public:
  static CopyPool &get() {
    static CopyPool *p = new CopyPool();  // never destroyed: its threads may outlive static objects
    return *p;
  }
  void copy(void *dst, const void *src, size_t n) {
    std::unique_lock<std::mutex> use(use_, std::try_to_lock);
    if (n < kMin || !use.owns_lock() || workers_ == 0) {
      std::memcpy(dst, src, n);
      return;
    }
    {
      std::lock_guard<std::mutex> lk(m_);
      dst_ = static_cast<uint8_t *>(dst);
      src_ = static_cast<const uint8_t *>(src);
      n_ = n;
      next_ = 0;
      done_ = 0;
      ++job_;
    }
    cv_.notify_all();
    work();
    // Blocks that a worker took are under way; the others the caller took.
    std::unique_lock<std::mutex> lk(m_);
    idle_.wait(lk, [&] { return done_ >= n_; });
    n_ = 0;
  }

 private:
  static constexpr size_t kMin = size_t(1) << 20, kBlock = size_t(256) << 10;
  CopyPool() {
    const unsigned cpus = std::thread::hardware_concurrency();
    const int want = (int)std::min(5u, cpus > 2 ? cpus / 2 : 0u);
    for (int i = 0; i < want; ++i) {
      try {
        std::thread(&CopyPool::loop, this).detach();
        ++workers_;
      } catch (...) {
        break;  // fewer threads, or none: the caller copies
      }
    }
  }
  // Takes blocks until none is left.
  void work() {
    for (;;) {
      uint8_t *d;
      const uint8_t *s;
      size_t k;
      {
        std::lock_guard<std::mutex> lk(m_);
        if (next_ >= n_) return;
        d = dst_ + next_;
        s = src_ + next_;
        k = std::min(kBlock, n_ - next_);
        next_ += k;
      }
      std::memcpy(d, s, k);
      std::lock_guard<std::mutex> lk(m_);
      done_ += k;
      if (done_ >= n_) idle_.notify_all();
    }
  }
  void loop() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(m_);
        cv_.wait(lk, [&] { return job_ != seen; });
        seen = job_;
      }
      work();
    }
  }
  std::mutex use_, m_;
  std::condition_variable cv_, idle_;
  uint8_t *dst_ = nullptr;
  const uint8_t *src_ = nullptr;
  size_t n_ = 0, next_ = 0, done_ = 0;
  uint64_t job_ = 0;
  int workers_ = 0;
};

// A pinned block and the events of its pieces.
struct PinBlock {
  static constexpr int kEvents = 8;
  uint8_t *p = nullptr;
  size_t n = 0;
  int dev = 0;
  hipEvent_t ev[kEvents] = {};
};

}  // namespace rai

#endif
