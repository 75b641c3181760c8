// Host threads that help a call to copy.  One thread copies what a device has just written to host memory at about 26 GB/s,
// first touches of fresh pages at 4: 12 rows of 65536 logits took 120 us behind their step, more than their way over PCIe.
#pragma once
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace gptoss {

// Belongs to one caller at a time.  The threads start with the first run and end with the crew; while there is nothing to do
// they sleep (after a job they look for the next one for some 50 us: a result comes in two halves).
class CopyCrew {
 public:
  CopyCrew() = default;
  CopyCrew(const CopyCrew &) = delete;
  ~CopyCrew() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      stop_ = true;
      round_.fetch_add(1);
    }
    wake_.notify_all();
    for (std::thread &t : threads_) t.join();
  }

  // f(i) for every i < n, by this thread and those that wake in time; returns when all are done.
  template <typename F>
  void run(int n, const F &f) {
    start();
    {
      std::lock_guard<std::mutex> lock(mu_);
      call_ = [](const void *g, int i) { (*static_cast<const F *>(g))(i); };
      job_ = &f;
      n_ = n;
      next_.store(0);
      open_ = true;
      round_.fetch_add(1);
    }
    wake_.notify_all();
    work();
    std::unique_lock<std::mutex> lock(mu_);
    open_ = false;   // who wakes from now on finds nothing
    done_.wait(lock, [this] { return active_ == 0; });
  }

 private:
  static constexpr int HELPERS = 3;

  void start() {
    if (started_) return;
    started_ = true;
    try {
      for (int i = 0; i < HELPERS; i++) threads_.emplace_back([this] { serve(); });
    } catch (...) {   // no more threads to be had: the caller copies with those there are, or alone
    }
  }
  void work() {
    for (int i; (i = next_.fetch_add(1)) < n_;) call_(job_, i);
  }
  void serve() {
    unsigned long long seen = 0;
    for (;;) {
      for (int spin = 0; spin < 1500 && seen && round_.load() == seen; spin++) __builtin_ia32_pause();
      std::unique_lock<std::mutex> lock(mu_);
      wake_.wait(lock, [&] { return stop_ || round_.load() != seen; });
      if (stop_) return;
      seen = round_.load();
      if (!open_) continue;
      active_++;
      lock.unlock();
      work();
      lock.lock();
      if (--active_ == 0) done_.notify_one();
    }
  }

  std::mutex mu_;
  std::condition_variable wake_, done_;
  std::vector<std::thread> threads_;
  std::atomic<unsigned long long> round_{0};   // of jobs
  std::atomic<int> next_{0};
  void (*call_)(const void *, int) = nullptr;
  const void *job_ = nullptr;
  int n_ = 0, active_ = 0;
  bool open_ = false, stop_ = false, started_ = false;
};

}  // namespace gptoss
