#include "parallel.h"

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <deque>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>

namespace arb {

struct BackgroundTasks::Job {
  std::function<void(size_t)> fn;
  size_t n = 0;
  std::atomic<size_t> next{0};
  std::atomic<bool> stop{false};  // a task has thrown: the ones not started are left out
  std::mutex mutex;
  std::condition_variable all_done;
  size_t done = 0;
  std::exception_ptr failed;

  bool Exhausted() const { return next.load(std::memory_order_relaxed) >= n; }
  // runs tasks until none is left
  void Work() {
    size_t mine = 0;
    for (size_t i = next++; i < n; i = next++) {
      ++mine;
      if (stop) continue;
      try {
        fn(i);
      } catch (...) {
        std::lock_guard<std::mutex> lock(mutex);
        if (!failed) failed = std::current_exception();
        stop = true;
      }
    }
    if (mine == 0) return;
    std::lock_guard<std::mutex> lock(mutex);
    done += mine;
    if (done == n) all_done.notify_all();
  }
  void Wait() {
    Work();
    std::unique_lock<std::mutex> lock(mutex);
    all_done.wait(lock, [&] { return done == n; });
  }
};

// Workers that sleep until a job has tasks left.  Never destroyed: they may be asleep when the
// process ends.
class ThreadPool {
 public:
  using Job = BackgroundTasks::Job;
  explicit ThreadPool(size_t workers) : workers_(workers) {
    for (size_t t = 0; t < workers; ++t) std::thread([this] { Loop(); }).detach();
  }
  size_t workers() const { return workers_; }
  void Add(const std::shared_ptr<Job> &job) {
    const size_t helpers = std::min(workers_, job->n);
    {
      std::lock_guard<std::mutex> lock(mutex_);
      jobs_.push_back(job);
    }
    if (helpers >= workers_ / 2) wake_.notify_all();
    else
      for (size_t k = 0; k < helpers; ++k) wake_.notify_one();
  }

  // The pool of this process (a child made by fork has none of its parent's threads).
  static ThreadPool &Get() {
    static std::mutex guard;
    static ThreadPool *pool = nullptr;
    static pid_t owner = 0;
    std::lock_guard<std::mutex> lock(guard);
    if (!pool || owner != getpid()) {
      const size_t hw = std::max<size_t>(1, std::thread::hardware_concurrency());
      pool = new ThreadPool(std::min<size_t>(hw, 16) - 1);
      owner = getpid();
    }
    return *pool;
  }

 private:
  void Loop() {
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
      while (!jobs_.empty() && jobs_.front()->Exhausted()) jobs_.pop_front();
      if (jobs_.empty()) {
        wake_.wait(lock);
        continue;
      }
      std::shared_ptr<Job> job = jobs_.front();
      lock.unlock();
      job->Work();
      job.reset();
      lock.lock();
    }
  }
  const size_t workers_;
  std::mutex mutex_;
  std::condition_variable wake_;
  std::deque<std::shared_ptr<Job>> jobs_;
};

BackgroundTasks::~BackgroundTasks() {
  if (job_) job_->Wait();
}

void BackgroundTasks::Start(size_t n, std::function<void(size_t)> fn) {
  Wait();
  if (n == 0) return;
  job_ = std::make_shared<Job>();
  job_->fn = std::move(fn);
  job_->n = n;
  ThreadPool::Get().Add(job_);
}

void BackgroundTasks::Wait() {
  if (!job_) return;
  const std::shared_ptr<Job> job = std::move(job_);
  job_.reset();
  job->Wait();
  if (job->failed) std::rethrow_exception(job->failed);
}

void ParallelTasks(size_t n, const std::function<void(size_t)> &fn) {
  if (n == 0) return;
  if (n == 1 || ThreadPool::Get().workers() == 0) {
    for (size_t i = 0; i < n; ++i) fn(i);
    return;
  }
  BackgroundTasks tasks;
  tasks.Start(n, fn);
  tasks.Wait();
}

void ParallelFor(size_t n, const std::function<void(size_t, size_t)> &fn, size_t grain) {
  if (n == 0) return;
  const size_t threads = 16;
  // up to four pieces per thread, so that a thread that starts late does not hold up the loop
  const size_t pieces = std::min(n / std::max<size_t>(grain, 1), 4 * threads);
  if (pieces < 2) {
    fn(0, n);
    return;
  }
  const size_t chunk = (n + pieces - 1) / pieces;
  ParallelTasks((n + chunk - 1) / chunk, [&](size_t t) { fn(t * chunk, std::min(n, (t + 1) * chunk)); });
}

}  // namespace arb
