#include "memory_pool.h"

#include <hip/hip_runtime.h>
#include <unistd.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <map>
#include <mutex>
#include <new>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

namespace arb {
namespace {

constexpr size_t kDevicePoolBytes = (size_t)16 << 30;  // of 288 GB
constexpr size_t kPinnedPoolBytes = (size_t)256 << 20;
constexpr size_t kHostPoolBytes = (size_t)1 << 30;
constexpr double kPoolIdleSeconds = 60.0;

using Clock = std::chrono::steady_clock;

// Sizes are rounded up so that objects of similar size share blocks: to 512 bytes, from 4 KB on to
// an eighth of the largest power of two below.
size_t RoundSize(size_t bytes) {
  size_t step = 512;
  while (step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

class Pool {
 public:
  typedef void *(*Alloc)(size_t);  // null: no memory
  typedef void (*Free)(void *);
  Pool(Alloc alloc, Free free, size_t most) : alloc_(alloc), free_(free), most_(most) {}

  void *Take(int device, size_t bytes) {
    const size_t size = RoundSize(bytes < 1 ? 1 : bytes);
    std::lock_guard<std::mutex> lock(mutex_);
    DropOld();
    // the smallest idle block that fits and wastes less than a quarter
    auto it = idle_.lower_bound(Key{device, size});
    if (it != idle_.end() && it->first.device == device && it->first.size <= size + size / 4) {
      void *p = it->second.p;
      used_[p] = it->first;
      idle_bytes_ -= it->first.size;
      idle_.erase(it);
      return p;
    }
    void *p = alloc_(size);
    if (!p) {
      DropAll(device);
      p = alloc_(size);
    }
    if (p) used_[p] = Key{device, size};
    return p;
  }

  void Give(void *p) noexcept {
    if (!p) return;
    try {
      std::lock_guard<std::mutex> lock(mutex_);
      auto it = used_.find(p);
      if (it == used_.end()) return;
      const Key key = it->second;
      used_.erase(it);
      if (key.size > most_) {
        free_(p);
        return;
      }
      idle_.emplace(key, Idle{p, Clock::now()});
      idle_bytes_ += key.size;
      while (idle_bytes_ > most_) DropOldest();
      DropOld();
    } catch (...) {  // (no memory for the bookkeeping)
      free_(p);
    }
  }

  void Trim(int device) noexcept {
    std::lock_guard<std::mutex> lock(mutex_);
    DropAll(device);
  }
  void TrimAll() noexcept {
    std::lock_guard<std::mutex> lock(mutex_);
    while (!idle_.empty()) Drop(idle_.begin());
  }

 private:
  struct Key {
    int device;
    size_t size;
    bool operator<(const Key &o) const { return device != o.device ? device < o.device : size < o.size; }
  };
  struct Idle {
    void *p;
    Clock::time_point since;
  };

  void Drop(std::multimap<Key, Idle>::iterator it) {
    free_(it->second.p);
    idle_bytes_ -= it->first.size;
    idle_.erase(it);
  }
  void DropOldest() {
    auto oldest = idle_.begin();
    for (auto it = idle_.begin(); it != idle_.end(); ++it)
      if (it->second.since < oldest->second.since) oldest = it;
    Drop(oldest);
  }
  void DropOld() {
    const Clock::time_point now = Clock::now();
    if (std::chrono::duration<double>(now - looked_).count() < kPoolIdleSeconds / 4) return;
    looked_ = now;
    for (auto it = idle_.begin(); it != idle_.end();) {
      auto next = std::next(it);
      if (std::chrono::duration<double>(now - it->second.since).count() > kPoolIdleSeconds) Drop(it);
      it = next;
    }
  }
  void DropAll(int device) {
    for (auto it = idle_.begin(); it != idle_.end();) {
      auto next = std::next(it);
      if (it->first.device == device) Drop(it);
      it = next;
    }
  }

  const Alloc alloc_;
  const Free free_;
  const size_t most_;
  std::mutex mutex_;
  std::multimap<Key, Idle> idle_;
  std::unordered_map<void *, Key> used_;
  size_t idle_bytes_ = 0;
  Clock::time_point looked_ = Clock::now();
};

// The pools live until the process ends (a block may be given back by a destructor that runs at its
// very end, when the driver may be gone: nothing is freed there).
Pool &DevicePool() {
  static Pool *p = new Pool(
      [](size_t n) -> void * {
        void *q = nullptr;
        if (hipMalloc(&q, n) != hipSuccess) {
          (void)hipGetLastError();  // (the error is reported by Take, not by the next launch)
          return nullptr;
        }
        return q;
      },
      [](void *q) { (void)hipFree(q); }, kDevicePoolBytes);
  return *p;
}
Pool &PinnedPool() {
  static Pool *p = new Pool(
      [](size_t n) -> void * {
        void *q = nullptr;
        if (hipHostMalloc(&q, n, hipHostMallocDefault) != hipSuccess) {
          (void)hipGetLastError();
          return nullptr;
        }
        return q;
      },
      [](void *q) { (void)hipHostFree(q); }, kPinnedPoolBytes);
  return *p;
}
Pool &HostPool() {
  static Pool *p = new Pool([](size_t n) -> void * { return std::aligned_alloc(4096, (n + 4095) / 4096 * 4096); },
                            [](void *q) { std::free(q); }, kHostPoolBytes);
  return *p;
}

int CurrentDevice() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) (void)hipGetLastError();
  return dev;
}

std::atomic<pid_t> g_gpu_user{0};
void NoteGpuInUse() { g_gpu_user.store(getpid(), std::memory_order_relaxed); }

}  // namespace

bool GpuInUse() noexcept { return g_gpu_user.load(std::memory_order_relaxed) == getpid(); }

void *DevicePoolTake(size_t bytes) {
  void *p = DevicePool().Take(CurrentDevice(), bytes);
  if (p) NoteGpuInUse();
  if (!p) throw std::runtime_error("HIP error: out of memory allocating " + std::to_string(bytes) + " bytes of device memory");
  return p;
}
void DevicePoolGive(void *p) noexcept { DevicePool().Give(p); }
void DevicePoolTrim() noexcept { DevicePool().Trim(CurrentDevice()); }

namespace {
constexpr size_t kIdleStreams = 16;
std::mutex g_streams_mutex;
struct Streams {
  std::vector<std::pair<int, hipStream_t>> idle;
  std::unordered_map<hipStream_t, int> made_on;  // the device of every stream, in use or idle
};
Streams &PooledStreams() {
  static auto *v = new Streams();
  return *v;
}
}  // namespace

hipStream_t StreamPoolTake() {
  const int dev = CurrentDevice();
  {
    std::lock_guard<std::mutex> lock(g_streams_mutex);
    auto &idle = PooledStreams().idle;
    for (size_t k = 0; k < idle.size(); ++k)
      if (idle[k].first == dev) {
        hipStream_t s = idle[k].second;
        idle.erase(idle.begin() + k);
        NoteGpuInUse();
        return s;
      }
  }
  hipStream_t s = nullptr;
  const hipError_t e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
  if (e != hipSuccess) throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e) + " creating a stream");
  try {
    std::lock_guard<std::mutex> lock(g_streams_mutex);
    PooledStreams().made_on[s] = dev;
  } catch (...) {
    (void)hipStreamDestroy(s);
    throw;
  }
  NoteGpuInUse();
  return s;
}

void StreamPoolGive(hipStream_t s) noexcept {
  if (!s) return;
  {
    std::lock_guard<std::mutex> lock(g_streams_mutex);
    // back to the device it was made on: the thread that gives it may use another one
    auto &pool = PooledStreams();
    const auto it = pool.made_on.find(s);
    if (it != pool.made_on.end() && pool.idle.size() < kIdleStreams) {
      try {
        pool.idle.emplace_back(it->second, s);
        return;
      } catch (...) {
      }
    }
    if (it != pool.made_on.end()) pool.made_on.erase(it);
  }
  (void)hipStreamDestroy(s);
}

void *PinnedPoolTake(size_t bytes) {
  void *p = PinnedPool().Take(0, bytes);
  if (!p) throw std::runtime_error("HIP error: out of memory allocating " + std::to_string(bytes) + " bytes of pinned host memory");
  return p;
}
void PinnedPoolGive(void *p) noexcept { PinnedPool().Give(p); }

void *HostPoolTake(size_t bytes) {
  void *p = HostPool().Take(0, bytes);
  if (!p) throw std::bad_alloc();
  return p;
}
void HostPoolGive(void *p) noexcept { HostPool().Give(p); }

void TrimPools() noexcept {
  HostPool().TrimAll();
  if (!GpuInUse()) return;  // (what a parent's pools held is not a child's to free)
  DevicePool().TrimAll();
  PinnedPool().TrimAll();
  std::lock_guard<std::mutex> lock(g_streams_mutex);
  auto &pool = PooledStreams();
  for (const auto &s : pool.idle) {
    pool.made_on.erase(s.second);
    (void)hipStreamDestroy(s.second);
  }
  pool.idle.clear();
}

}  // namespace arb
