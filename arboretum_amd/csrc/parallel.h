// Host threads for the library's own loops.
#ifndef ARBORETUM_AMD_PARALLEL_H_
#define ARBORETUM_AMD_PARALLEL_H_

#include <cstddef>
#include <functional>
#include <memory>

namespace arb {

// fn(begin, end) over [0, n) in pieces of at least `grain` items, on the calling thread and up to
// 15 workers that are started once and kept (starting sixteen threads takes longer than most of
// the loops here run).  The first exception of any piece is handed back to the caller.
void ParallelFor(size_t n, const std::function<void(size_t, size_t)> &fn, size_t grain = 16384);
// fn(i) for every i in [0, n), a few long tasks (columns) handed out one at a time.
void ParallelTasks(size_t n, const std::function<void(size_t)> &fn);

// A few long tasks that run beside the caller (filling the next staging buffer while the GPU works
// on the previous one).  Wait() helps with what has not been started and rethrows; the destructor
// waits as well, so that what the tasks refer to may be a local of the caller.
class BackgroundTasks {
 public:
  BackgroundTasks() {}
  ~BackgroundTasks();
  BackgroundTasks(const BackgroundTasks &) = delete;
  BackgroundTasks &operator=(const BackgroundTasks &) = delete;
  void Start(size_t n, std::function<void(size_t)> fn);  // waits for the tasks of the call before
  void Wait();

 private:
  struct Job;
  friend class ThreadPool;
  friend void ParallelTasks(size_t, const std::function<void(size_t)> &);
  std::shared_ptr<Job> job_;
};

}  // namespace arb
#endif  // ARBORETUM_AMD_PARALLEL_H_
