// The pools of memory and streams (memory_pool.h) over the runtime of fake_hip.h.
#include <cstdio>
#include <cstring>
#include <set>
#include <thread>
#include <vector>

#include "../../arboretum_amd/csrc/memory_pool.h"
#include "fake_hip.h"

#define CHECK(x)                                                    \
  do {                                                              \
    if (!(x)) {                                                     \
      std::printf("%s:%d: %s is false\n", __FILE__, __LINE__, #x);  \
      return 1;                                                     \
    }                                                               \
  } while (0)

// What was taken on one device goes back to it, whichever device is current when it is given back.
int OtherDevice() {
  fake::current = 1;
  std::vector<hipStream_t> streams;
  for (int k = 0; k < 20; ++k) streams.push_back(arb::StreamPoolTake());
  void *block = arb::DevicePoolTake(1 << 20);
  std::thread([&] {  // (device 0 is current there)
    for (hipStream_t s : streams) arb::StreamPoolGive(s);
    arb::DevicePoolGive(block);
  }).join();
  for (int device : {0, 1, 0, 1}) {
    fake::current = device;
    std::vector<hipStream_t> taken;
    for (int k = 0; k < 20; ++k) {
      taken.push_back(arb::StreamPoolTake());
      CHECK(fake::streams.at(taken.back()) == device);
    }
    void *p = arb::DevicePoolTake(1 << 20);
    CHECK(fake::blocks.at(p).first == device);
    fake::current = 1 - device;
    for (hipStream_t s : taken) arb::StreamPoolGive(s);
    arb::DevicePoolGive(p);
  }
  CHECK(fake::streams.size() <= 16);  // (no more idle ones are kept)
  return 0;
}

// Threads that take and give at the same time never hold the same block or stream.
int Threads() {
  std::vector<std::thread> threads;
  std::mutex mutex;
  std::set<void *> held;
  bool twice = false;
  for (int t = 0; t < 8; ++t)
    threads.emplace_back([&, t] {
      fake::current = t & 1;
      for (int k = 0; k < 2000; ++k) {
        void *p = arb::DevicePoolTake(4096 * (1 + (k + t) % 3));
        void *s = arb::StreamPoolTake();
        {
          std::lock_guard<std::mutex> lock(mutex);
          twice = twice || !held.insert(p).second || !held.insert(s).second;
        }
        std::lock_guard<std::mutex> lock(mutex);
        held.erase(p);
        held.erase(s);
        arb::DevicePoolGive(p);
        arb::StreamPoolGive(static_cast<hipStream_t>(s));
      }
    });
  for (auto &t : threads) t.join();
  CHECK(!twice);
  return 0;
}

// Idle blocks are bounded, and make room when the device is full.
int Bounds() {
  fake::current = 2;
  std::vector<void *> p;
  for (int k = 0; k < 20; ++k) p.push_back(arb::DevicePoolTake((size_t)1 << 30));
  for (void *q : p) arb::DevicePoolGive(q);
  CHECK(fake::BytesOn(2) <= (size_t)16 << 30);
  const size_t idle = fake::BytesOn(2);
  CHECK(idle >= (size_t)15 << 30);
  fake::capacity = idle + ((size_t)1 << 30);
  void *q = arb::DevicePoolTake((size_t)3 << 30);  // fits only when idle blocks go
  CHECK(fake::BytesOn(2) <= fake::capacity);
  bool refused = false;
  try {
    arb::DevicePoolTake(fake::capacity + 1);
  } catch (const std::exception &) {
    refused = true;
  }
  CHECK(refused);
  arb::DevicePoolGive(q);
  arb::DevicePoolTrim();
  CHECK(fake::BytesOn(2) == 0);
  fake::capacity = (size_t)1 << 40;
  return 0;
}

// TrimPools gives back everything idle, of every device, and nothing in use.
int Release() {
  void *kept[3];
  hipStream_t stream[3];
  for (int device = 0; device < 3; ++device) {
    fake::current = device;
    kept[device] = arb::DevicePoolTake(1 << 16);
    stream[device] = arb::StreamPoolTake();
    arb::DevicePoolGive(arb::DevicePoolTake(1 << 20));
    arb::PinnedPoolGive(arb::PinnedPoolTake(1 << 20));
    hipStream_t other = arb::StreamPoolTake();
    arb::StreamPoolGive(other);
  }
  CHECK(fake::blocks.size() == 6 && fake::streams.size() == 6 && fake::pinned.size() == 1);
  arb::TrimPools();
  CHECK(fake::blocks.size() == 3 && fake::streams.size() == 3 && fake::pinned.empty());
  for (int device = 0; device < 3; ++device) {
    CHECK(fake::blocks.count(kept[device]) && fake::streams.count(stream[device]));
    arb::DevicePoolGive(kept[device]);
    arb::StreamPoolGive(stream[device]);
  }
  arb::TrimPools();
  CHECK(fake::blocks.empty() && fake::streams.empty());
  return 0;
}

int main(int, char **argv) {
  if (!std::strcmp(argv[1], "other_device")) return OtherDevice();
  if (!std::strcmp(argv[1], "threads")) return Threads();
  if (!std::strcmp(argv[1], "bounds")) return Bounds();
  if (!std::strcmp(argv[1], "release")) return Release();
  return 2;
}
