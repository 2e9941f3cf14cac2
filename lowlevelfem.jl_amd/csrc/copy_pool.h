// The threads that empty pinned staging slots into a caller's memory
// (copy_to_host).  Host code only.
#pragma once

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>

namespace llfem {

// Up to eight threads, each its slice of every chunk.  They belong to one
// context (whose calls one host thread makes), which joins them.  A thread
// that waits for a chunk spins for kSpin and sleeps beyond that: the next chunk
// of a copy under way is 70 us (4 MB) or more away, but what a stream still has
// to do before the copy, or between two parts of it, can take milliseconds.  A
// thread woken late costs the copy 20 us.  Spinning for 20, 100, 200 us, without
// end: 2.1 MB 88, 67, 68, 71 us, 3.7 MB 120, 101, 101, 106 us; CPU time of a
// 248 MB copy (4.69 ms) 22, 33, 41, 42 ms.
class CopyPool {
 public:
  static constexpr int kSlots = 8;
  static constexpr int kThreads = 8;
  static constexpr std::chrono::microseconds kSpin{100};

  CopyPool() {
    const unsigned want = std::max(1u, std::min((unsigned)kThreads, std::thread::hardware_concurrency()));
    try {
      for (unsigned t = 0; t < want; ++t) {
        th_[n_] = std::thread([this, t] { run((int)t); });
        ++n_;
      }
    } catch (...) {   // fewer threads; none at all: the caller copies
    }
  }
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      quit_ = true;
    }
    cv_.notify_all();
    for (int t = 0; t < n_; ++t) th_[t].join();
  }
  int threads() const { return n_; }
  // A copy of `chunks` chunks by `use` of the threads, chunk i staged in slot
  // i % kSlots; arrived() hands one over, wait_free() returns when slot s is
  // empty again, finish() when every chunk given is copied (abandon: without
  // the others).
  void begin(size_t chunks, int use) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      use_ = std::max(1, std::min(use, n_));
      chunks_ = chunks;
      ready_.store(0);
      abandon_.store(false);
      for (auto& d : left_) d.store(0);
      active_.store(use_);
      ++gen_;
    }
    cv_.notify_all();
  }
  void arrived(size_t i, char* dst, const char* src, size_t len) {
    Part& p = part_[i % kSlots];
    p.dst = dst;
    p.src = src;
    p.len = len;
    left_[i % kSlots].store(use_);
    signal([&] { ready_.store(i + 1, std::memory_order_release); });
  }
  void wait_free(size_t s) {
    while (left_[s].load(std::memory_order_acquire) > 0) std::this_thread::yield();
  }
  void finish(bool abandon) {
    if (abandon) signal([&] { abandon_.store(true); });
    while (active_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
  }

 private:
  struct Part {
    char* dst;
    const char* src;
    size_t len;
  };
  // A change that a thread may sleep for: made under the lock, so that none
  // goes to sleep between its last look and the notification.
  template <typename F>
  void signal(F change) {
    bool wake;
    {
      std::lock_guard<std::mutex> lk(mu_);
      change();
      wake = asleep_ > 0;
    }
    if (wake) cv_.notify_all();
  }
  bool due(size_t i) const {
    return ready_.load(std::memory_order_acquire) > i || abandon_.load(std::memory_order_acquire);
  }
  // Returns when chunk i is there (true) or the copy is abandoned without it.
  bool wait_chunk(size_t i) {
    const auto t0 = std::chrono::steady_clock::now();
    for (int spin = 0; !due(i);) {
      if (++spin < 2000) continue;
      if (std::chrono::steady_clock::now() - t0 < kSpin) {
        std::this_thread::yield();
        continue;
      }
      std::unique_lock<std::mutex> lk(mu_);
      ++asleep_;
      cv_.wait(lk, [&] { return due(i); });
      --asleep_;
    }
    return ready_.load(std::memory_order_acquire) > i;
  }
  void run(int t) {
    uint64_t seen = 0;
    for (;;) {
      size_t chunks;
      int use;
      {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return quit_ || (gen_ != seen && t < use_); });
        if (quit_) return;
        seen = gen_;
        chunks = chunks_;
        use = use_;
      }
      for (size_t i = 0; i < chunks && wait_chunk(i); ++i) {
        const Part p = part_[i % kSlots];
        const size_t per = ((p.len + use - 1) / use + 63) / 64 * 64;
        const size_t lo = std::min(p.len, t * per), hi = std::min(p.len, lo + per);
        if (lo < hi) std::memcpy(p.dst + lo, p.src + lo, hi - lo);
        left_[i % kSlots].fetch_sub(1, std::memory_order_release);
      }
      active_.fetch_sub(1, std::memory_order_release);
    }
  }
  std::thread th_[kThreads];
  int n_ = 0;
  std::mutex mu_;
  std::condition_variable cv_;
  uint64_t gen_ = 0;
  int use_ = 1, asleep_ = 0;
  bool quit_ = false;
  size_t chunks_ = 0;
  Part part_[kSlots] = {};
  std::atomic<size_t> ready_{0};
  std::atomic<int> left_[kSlots] = {};
  std::atomic<int> active_{0};
  std::atomic<bool> abandon_{false};
};

}  // namespace llfem
