// Host threads that copy and convert arrays beside the transfers.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace gcs {

// A persistent pool of host threads: run(n, fn) calls fn(begin, end) on
// disjoint ranges covering [0, n) and returns when all are done. Calls are
// serialised. Threads that the system does not grant are done without: callers
// are C entry points, which no exception may leave.
class HostPool {
 public:
  static HostPool &get() {
    static HostPool pool;
    return pool;
  }

  void run(long n, const std::function<void(long, long)> &fn) {
    std::lock_guard<std::mutex> serial(run_lock_);
    const long parts = std::min<long>(n, (long)workers_.size() + 1);
    if (parts <= 1) {
      if (n > 0) fn(0, n);
      return;
    }
    {
      std::unique_lock<std::mutex> lk(m_);
      fn_ = &fn;
      n_ = n;
      parts_ = parts;
      next_ = 1;  // part 0 runs on the calling thread
      done_ = 0;
      ++generation_;
    }
    cv_.notify_all();
    fn(0, n / parts);
    std::unique_lock<std::mutex> lk(m_);
    done_cv_.wait(lk, [&] { return done_ == parts_ - 1; });
    fn_ = nullptr;
  }

 private:
  HostPool() {
    const unsigned hw = std::thread::hardware_concurrency();
    const unsigned count = std::max(1u, std::min(16u, hw == 0 ? 1u : hw)) - 1;
    try {
      workers_.reserve(count);
      for (unsigned t = 0; t < count; ++t) workers_.emplace_back([this] { loop(); });
    } catch (const std::exception &) {  // the calling thread and those there are
    }
  }
  ~HostPool() {
    {
      std::lock_guard<std::mutex> lk(m_);
      stop_ = true;
    }
    cv_.notify_all();
    for (std::thread &t : workers_) t.join();
  }

  void loop() {
    unsigned long seen = 0;
    std::unique_lock<std::mutex> lk(m_);
    for (;;) {
      cv_.wait(lk, [&] { return stop_ || (generation_ != seen && next_ < parts_); });
      if (stop_) return;
      const long part = next_++;
      if (next_ >= parts_) seen = generation_;
      const std::function<void(long, long)> *fn = fn_;
      const long n = n_, parts = parts_;
      lk.unlock();
      (*fn)(n * part / parts, n * (part + 1) / parts);
      lk.lock();
      if (++done_ == parts_ - 1) done_cv_.notify_one();
    }
  }

  std::vector<std::thread> workers_;
  std::mutex run_lock_, m_;
  std::condition_variable cv_, done_cv_;
  const std::function<void(long, long)> *fn_ = nullptr;
  long n_ = 0, parts_ = 0, next_ = 0, done_ = 0;
  unsigned long generation_ = 0;
  bool stop_ = false;
};

}  // namespace gcs
