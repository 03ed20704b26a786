#pragma once

#include <sys/types.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>

namespace vh {

// Host thread pools of the table builder and of the staged copies (transfer.hip): run(n, f) calls
// f(i) for i in [0, n) on the pool's workers and the caller, returning when all are done.
// Created on first use with min(hardware threads, 16) threads (VESPAHIP_HOST_THREADS
// overrides, 1 = serial), the copies' with kCopyThreads at most; a child process after fork() builds its own (it
// inherits no worker threads). Where the system gives fewer threads the pool has
// fewer, down to the caller alone. The pool is never destroyed: its workers sleep
// until the process ends.
class HostPool {
 public:
  static int threads() {
    static const int n = [] {
      const char* e = getenv("VESPAHIP_HOST_THREADS");
      int v = e ? atoi(e) : (int)std::thread::hardware_concurrency();
      return std::max(1, std::min(v, e ? 256 : 16));
    }();
    return n;
  }
  static void run(int n, const std::function<void(int)>& f) {
    static HostPool* pool = nullptr;
    run_on(pool, threads(), n, f);
  }
  static void run_copies(int n, const std::function<void(int)>& f) {
    static HostPool* pool = nullptr;
    run_on(pool, std::min(threads(), kCopyThreads), n, f);
  }

 private:
  // Four threads copy at the link's rate (down 200 MiB 5.9, 4.9, 4.3 and 4.3 ms with 2, 3, 4 and 16), fault
  // a fresh array's huge pages with less contention (10.7 ms with 4, 13.9 with 16), and leave
  // processors to the runtime's own threads while they spin (the hipFree after a copy 95 µs, 400 with
  // 16 on 16 processors).
  static constexpr int kCopyThreads = 4;

  static void run_on(HostPool*& pool, int nthreads, int n, const std::function<void(int)>& f) {
    if (n <= 1 || nthreads <= 1) {
      for (int i = 0; i < n; ++i) f(i);
      return;
    }
    static std::mutex create_mu;
    HostPool* p;
    {
      std::lock_guard<std::mutex> lk(create_mu);
      if (!pool || pool->pid_ != getpid()) pool = new HostPool(nthreads - 1);   // the old one stays (forked child)
      p = pool;
    }
    p->go(n, f);
  }

  // A build issues a few jobs back to back: threads spin this many pauses
  // (tens of microseconds) for the next job or the end of the current one
  // before they sleep, which saves a wake-up per job.
  static constexpr int kSpin = 1 << 14;
  static void pause() { __builtin_ia32_pause(); }

  explicit HostPool(int workers) : pid_(getpid()) {
    try {
      for (; nworkers_ < workers; ++nworkers_) std::thread([this] { loop(); }).detach();
    } catch (const std::system_error&) {
    }
  }
  void loop() {
    long long seen = 0;
    for (;;) {
      long long g = gen_.load(std::memory_order_acquire);
      for (int i = 0; g == seen && i < kSpin; ++i) {
        pause();
        g = gen_.load(std::memory_order_acquire);
      }
      if (g == seen) {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return gen_.load(std::memory_order_acquire) != seen; });
        g = gen_.load(std::memory_order_acquire);
      }
      seen = g;
      const std::function<void(int)>* f = job_;
      const int n = njob_;
      for (int i; (i = next_.fetch_add(1)) < n;) (*f)(i);
      if (active_.fetch_sub(1, std::memory_order_acq_rel) == 1) {
        std::lock_guard<std::mutex> lk(mu_);
        done_.notify_one();
      }
    }
  }
  void go(int n, const std::function<void(int)>& f) {
    std::lock_guard<std::mutex> run_lk(run_mu_);   // one job at a time
    job_ = &f;
    njob_ = n;
    next_.store(0);
    active_.store(nworkers_);
    {
      std::lock_guard<std::mutex> lk(mu_);
      gen_.fetch_add(1, std::memory_order_release);   // publishes the job to spinning and sleeping workers
    }
    cv_.notify_all();
    for (int i; (i = next_.fetch_add(1)) < n;) f(i);
    for (int i = 0; active_.load(std::memory_order_acquire) != 0 && i < kSpin; ++i) pause();
    if (active_.load(std::memory_order_acquire) != 0) {
      std::unique_lock<std::mutex> lk(mu_);
      done_.wait(lk, [&] { return active_.load(std::memory_order_acquire) == 0; });
    }
  }
  pid_t pid_;
  int nworkers_ = 0;
  std::mutex run_mu_, mu_;
  std::condition_variable cv_, done_;
  const std::function<void(int)>* job_ = nullptr;
  int njob_ = 0;
  std::atomic<long long> gen_{0};
  std::atomic<int> next_{0}, active_{0};
};

}  // namespace vh
