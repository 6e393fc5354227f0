// copy_pool.h -- host threads that share the copies of a transfer (hostio.hip).
// Plain C++, without the device.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace qphix {

constexpr size_t HOST_SLICE = (size_t)256 << 10;  // a thread's share at a time

// Threads that share the copies of a transfer.  They sleep between transfers
// and poll for slices during one (open).  The caller copies as well, so a pool of
// fewer threads than asked for, or of none, still completes every copy.
class CopyPool {
 public:
  explicit CopyPool(int workers) {
    try {
      for (int k = 0; k < workers; ++k) th_.emplace_back([this] { work(); });
    } catch (const std::exception &) {
      // no more threads to be had: the ones that started share the copies
    }
  }
  ~CopyPool() {  // also during a transfer, whose caller is leaving the process
    {
      std::lock_guard<std::mutex> l(m_);
      quit_ = true;
      open_.store(false);
    }
    cv_.notify_all();
    for (auto &t : th_) t.join();
  }
  void open() {
    {
      std::lock_guard<std::mutex> l(m_);
      open_.store(true);
    }
    cv_.notify_all();
  }
  void close() { open_.store(false); }
  // d[0..n) = s[0..n), all of it done on return
  void copy(char *d, const char *s, size_t n) {
    {
      std::lock_guard<std::mutex> l(m_);
      d_ = d;
      s_ = s;
      n_ = n;
      at_ = 0;
      left_.store(n);
      more_.store(n != 0);
    }
    while (step()) {}
    while (left_.load(std::memory_order_acquire) != 0) relax();
  }

 private:
  static void relax() { __builtin_ia32_pause(); }
  // copies one slice; false when none is left to take
  bool step() {
    char *d;
    const char *s;
    size_t n;
    {
      std::lock_guard<std::mutex> l(m_);
      n = std::min(HOST_SLICE, n_ - at_);
      if (n == 0) return false;
      d = d_ + at_;
      s = s_ + at_;
      at_ += n;
      if (at_ == n_) more_.store(false);
    }
    std::memcpy(d, s, n);
    left_.fetch_sub(n, std::memory_order_release);
    return true;
  }
  void work() {
    for (;;) {
      {
        std::unique_lock<std::mutex> l(m_);
        cv_.wait(l, [this] { return quit_ || open_.load(); });
        if (quit_) return;
      }
      int idle = 0;
      while (open_.load(std::memory_order_relaxed)) {
        if (more_.load(std::memory_order_relaxed) && step()) {
          idle = 0;
        } else if (++idle < 2000) {
          relax();
        } else {
          std::this_thread::yield();
        }
      }
    }
  }

  std::mutex m_;
  std::condition_variable cv_;
  std::vector<std::thread> th_;
  bool quit_ = false;
  std::atomic<bool> open_{false};
  // the copy in progress (guarded by m_)
  char *d_ = nullptr;
  const char *s_ = nullptr;
  size_t n_ = 0, at_ = 0;
  std::atomic<size_t> left_{0};  // its bytes not copied yet
  std::atomic<bool> more_{false};  // it has bytes that no thread has taken
};

} // namespace qphix
