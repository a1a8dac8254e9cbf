// Host side of the model calls' transfers between pageable memory and the
// device: a few copy threads, and the bookkeeping of the pinned staging blocks
// (no HIP here, so that the host can test it alone).
//
// hipMemcpyAsync on pageable memory moved 16.8 MB of hidden states at 12 to 15
// GB/s and took 30 to 70 us for a few kilobytes, each with a wait of its own
// (2.5 of the 6.5 ms of a 1024-token layer, half of a one-token layer).  Here a
// kernel reads or writes the pinned block directly (no copy engine hand-off),
// the host's copies run on several threads and overlap the device's piece by
// piece, and the call waits once.
#ifndef RAI_HOST_IO_H
#define RAI_HOST_IO_H

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

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

// At most Max blocks per device, in use and free together, for blocks that cost
// milliseconds to make.  Block has n (bytes) and dev.  Nothing here allocates or
// throws; making and freeing a block is the caller's.
enum class PoolTake {
  kBlock,    // b is a free block of n bytes or more
  kMake,     // none, but one more may be made: then give() it, or gone()
  kReplace,  // b is a smaller free block to drop for a new one: as kMake
  kNone      // Max are in use
};
template <class Block, int Max, int Devices = 64>
class BoundedPool {
 public:
  PoolTake take(size_t n, int dev, Block &b) noexcept {
    if (dev < 0 || dev >= Devices) return PoolTake::kNone;
    std::lock_guard<std::mutex> lk(m_);
    Slots &s = d_[dev];
    int best = -1;  // the smallest that fits
    for (int i = 0; i < s.nfree; ++i)
      if (s.free[i].n >= n && (best < 0 || s.free[i].n < s.free[best].n)) best = i;
    if (best < 0 && s.total < Max) {
      ++s.total;
      return PoolTake::kMake;
    }
    if (s.nfree == 0) return PoolTake::kNone;
    const int i = best < 0 ? 0 : best;
    b = s.free[i];
    s.free[i] = s.free[--s.nfree];
    return best < 0 ? PoolTake::kReplace : PoolTake::kBlock;
  }
  // The caller's block is free again.
  void give(const Block &b) noexcept {
    std::lock_guard<std::mutex> lk(m_);
    Slots &s = d_[b.dev];
    s.free[s.nfree++] = b;
  }
  // A block of the device was dropped, or not made after kMake or kReplace.
  void gone(int dev) noexcept {
    std::lock_guard<std::mutex> lk(m_);
    --d_[dev].total;
  }

 private:
  struct Slots {
    Block free[Max];
    int nfree = 0, total = 0;
  };
  std::mutex m_;
  Slots d_[Devices];
};

// At most Max free blocks kept for later calls, of any device; a block in use is
// its caller's alone.  Nothing here allocates or throws.
template <class Block, int Max>
class KeptBlocks {
 public:
  // The smallest kept block of dev with n bytes or more.
  bool take(size_t n, int dev, Block &b) noexcept {
    std::lock_guard<std::mutex> lk(m_);
    int best = -1;
    for (int i = 0; i < n_; ++i)
      if (k_[i].dev == dev && k_[i].n >= n && (best < 0 || k_[i].n < k_[best].n)) best = i;
    return best >= 0 && leave(best, b);
  }
  // Keeps b.  True when one is too many: the oldest leaves in `out`.
  bool keep(const Block &b, Block &out) noexcept {
    std::lock_guard<std::mutex> lk(m_);
    const bool full = n_ == Max && leave(0, out);
    k_[n_++] = b;
    return full;
  }
  // Any kept block of dev leaves.
  bool drop(int dev, Block &out) noexcept {
    std::lock_guard<std::mutex> lk(m_);
    for (int i = 0; i < n_; ++i)
      if (k_[i].dev == dev) return leave(i, out);
    return false;
  }

 private:
  bool leave(int i, Block &out) noexcept {
    out = k_[i];
    --n_;
    for (; i < n_; ++i) k_[i] = k_[i + 1];
    return true;
  }
  std::mutex m_;
  Block k_[Max];
  int n_ = 0;
};

}  // namespace rai

#endif
