// Host threads that move results and uploads between pinned staging and the
// caller's arrays.
//
// A copy straight from device memory into a pageable array runs at a few GB/s:
// the runtime pins or stages it on one thread, and a fresh array takes a page
// fault per 4 KiB on that thread.  Here the device copies into the context's
// pinned staging chunk by chunk and these threads move each finished chunk on
// (and take its page faults) while the next ones arrive.
#pragma once

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace llgpu {

class CopyPool {
 public:
  // At most kThreads workers besides the calling thread, started on first use
  // and joined by the destructor.  One caller at a time (as the context).
  static constexpr unsigned kThreads = 7;

  CopyPool() = default;
  CopyPool(const CopyPool&) = delete;
  CopyPool& operator=(const CopyPool&) = delete;
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
  }

  // Runs task(0) .. task(n - 1) on the workers and, once `lead` has returned,
  // on the calling thread; returns when all are done.  Neither may throw.
  // Without workers (none could be started) the caller runs every task.
  template <typename Lead>
  void run(size_t n, const std::function<void(size_t)>& task, Lead&& lead) {
    if (n > 1) start();
    if (n <= 1 || threads_.empty()) {
      lead();
      for (size_t i = 0; i < n; i++) task(i);
      return;
    }
    {
      std::lock_guard<std::mutex> lk(mu_);
      task_ = &task;
      n_ = n;
      next_.store(0);
      busy_ = unsigned(threads_.size());
      round_++;
    }
    cv_.notify_all();
    lead();
    work();
    std::unique_lock<std::mutex> lk(mu_);
    done_cv_.wait(lk, [&] { return busy_ == 0; });
    task_ = nullptr;
  }

 private:
  void start() {
    if (!threads_.empty()) return;
    const unsigned hw = std::thread::hardware_concurrency();
    const unsigned want = hw > 1 ? (hw - 1 < kThreads ? hw - 1 : kThreads) : 0;
    try {
      threads_.reserve(want);
      const uint64_t r = round_;
      for (unsigned i = 0; i < want; i++) threads_.emplace_back([this, r] { loop(r); });
    } catch (...) {  // fewer threads (or none) than wanted
    }
  }

  void work() {
    for (;;) {
      const size_t i = next_.fetch_add(1);
      if (i >= n_) return;
      (*task_)(i);
    }
  }

  void loop(uint64_t seen) {
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return stop_ || round_ != seen; });
        if (stop_) return;
        seen = round_;
      }
      work();
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (--busy_ == 0) done_cv_.notify_all();
      }
    }
  }

  std::vector<std::thread> threads_;
  std::mutex mu_;
  std::condition_variable cv_, done_cv_;
  const std::function<void(size_t)>* task_ = nullptr;
  size_t n_ = 0;
  std::atomic<size_t> next_{0};
  unsigned busy_ = 0;
  uint64_t round_ = 0;
  bool stop_ = false;
};

}  // namespace llgpu
