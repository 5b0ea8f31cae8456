// The rows of a matrix (float_rows.h) over the runtime of fake_hip.h: where they are kept, and from which device
// they are read.
#include <cstdio>
#include <cstring>
#include <numeric>
#include <thread>
#include <vector>

#include "../../arboretum_amd/csrc/float_rows.h"
#include "../../arboretum_amd/csrc/memory_pool.h"
#include "fake_hip.h"

#define CHECK(x)                                                    \
  do {                                                              \
    if (!(x)) {                                                     \
      std::printf("%s:%d: %s is false\n", __FILE__, __LINE__, #x);  \
      return 1;                                                     \
    }                                                               \
  } while (0)

static std::vector<float> Rows(size_t n) {
  std::vector<float> x(n);
  std::iota(x.begin(), x.end(), 1.0f);
  return x;
}
static void UseGpu() { arb::DevicePoolGive(arb::DevicePoolTake(1)); }

// Rows kept on device 1, asked for by a thread that uses device 0: not handed to its kernels, and fetched to the host by
// a stream of device 1.
int OtherDevice() {
  for (size_t columns : {70u, 3000u}) {  // a piece or two, and many
    const std::vector<float> x = Rows(1000 * columns);
    fake::current = 1;
    UseGpu();
    arb::FloatRows rows(x.data(), 1000, columns);
    CHECK(rows.OnDevice() != nullptr);
    fake::current = 0;
    CHECK(rows.OnDevice() == nullptr);
    const float *host = rows.OnHost();
    CHECK(host && !std::memcmp(host, x.data(), x.size() * sizeof(float)));
    CHECK(fake::current == 0);
    CHECK(rows.OnHost() == host);
  }
  return 0;
}

// A process that does not use the GPU keeps them on the host, and one whose device is full as well, until there is room.
int Places() {
  const std::vector<float> x = Rows(200000);
  arb::FloatRows early(x.data(), 2000, 100);
  CHECK(fake::blocks.empty() && fake::streams.empty());
  UseGpu();
  arb::FloatRows small(x.data(), 10, 100);  // pinned: kernels of every device read it there
  CHECK(small.OnDevice() == small.OnHost());
  arb::TrimPools();
  fake::capacity = 700000;
  arb::FloatRows late(x.data(), 2000, 100);
  CHECK(late.OnDevice() == nullptr && fake::blocks.empty());
  fake::capacity = 1 << 20;
  const float *p = late.OnDevice();
  CHECK(p && fake::blocks.size() == 1 && !std::memcmp(p, x.data(), x.size() * sizeof(float)));
  CHECK(early.OnDevice() == nullptr && !std::memcmp(early.OnHost(), x.data(), x.size() * sizeof(float)));
  return 0;
}

int main(int, char **argv) {
  if (!std::strcmp(argv[1], "other_device")) return OtherDevice();
  if (!std::strcmp(argv[1], "places")) return Places();
  return 2;
}
