// A few host threads that share a loop with the thread that runs it: tables on
// their way out are widened faster than one thread can.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace xted {

// Owned by one Context and used under its lock. Threads start with the first
// loop that wants them and end with the pool.
class HostPool {
 public:
  static constexpr int kThreads = 4;  // with the caller

  ~HostPool() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (std::thread& t : threads_) t.join();
  }

  // fn(i) for every i in [0, n), on the calling thread and the pool's.
  void run(int64_t n, const std::function<void(int64_t)>& fn) {
    if (n > 1) start();
    if (n <= 1 || threads_.empty()) {
      for (int64_t i = 0; i < n; ++i) fn(i);
      return;
    }
    {
      std::lock_guard<std::mutex> lk(mu_);
      fn_ = &fn;
      n_ = n;
      next_ = 0;
      busy_ = (int)threads_.size();
      ++round_;
    }
    cv_.notify_all();
    for (int64_t i; (i = next_++) < n;) fn(i);
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [&] { return busy_ == 0; });
    fn_ = nullptr;
  }

 private:
  void start() {
    if (started_) return;
    started_ = true;
    const int want = std::min<int>(kThreads, (int)std::thread::hardware_concurrency()) - 1;
    try {
      for (int k = 0; k < want; ++k) threads_.emplace_back([this] { work(); });
    } catch (const std::system_error&) {
      // As many as there are; none: the caller runs the loop alone.
    }
  }

  void work() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      cv_.wait(lk, [&] { return stop_ || round_ != seen; });
      if (stop_) return;
      seen = round_;
      const auto* fn = fn_;
      const int64_t n = n_;
      lk.unlock();
      for (int64_t i; (i = next_++) < n;) (*fn)(i);
      lk.lock();
      if (--busy_ == 0) done_.notify_one();
    }
  }

  std::mutex mu_;
  std::condition_variable cv_, done_;
  std::vector<std::thread> threads_;
  const std::function<void(int64_t)>* fn_ = nullptr;
  std::atomic<int64_t> next_{0};
  int64_t n_ = 0;
  int busy_ = 0;
  uint64_t round_ = 0;
  bool started_ = false, stop_ = false;
};

}  // namespace xted
