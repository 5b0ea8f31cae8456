#include "float_rows.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <stdexcept>

#include "memory_pool.h"
#include "parallel.h"
#include "staging.h"

namespace arb {
namespace {

constexpr size_t kPinnedRowsBytes = (size_t)256 << 10;
constexpr size_t kDeviceRowsBytes = (size_t)8 << 30;
constexpr size_t kAllDeviceRowsBytes = (size_t)32 << 30;

std::atomic<size_t> g_device_bytes{0};

int CurrentDevice() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) (void)hipGetLastError();
  return dev;
}

// Another device current while the object lives.
struct OnDeviceOf {
  explicit OnDeviceOf(int device) : before(CurrentDevice()) {
    if (device != before && hipSetDevice(device) != hipSuccess) throw std::runtime_error("HIP error: no such device");
  }
  ~OnDeviceOf() { (void)hipSetDevice(before); }
  const int before;
};

struct PooledStream {
  hipStream_t s = StreamPoolTake();
  ~PooledStream() { StreamPoolGive(s); }
};

}  // namespace

FloatRows::FloatRows(const float *rows, size_t n, size_t columns) : n_(n), columns_(columns) {
  const size_t count = n * columns, bytes = count * sizeof(float);
  if (count == 0) return;
  if (GpuInUse()) {
    if (bytes <= kPinnedRowsBytes) {
      pinned_ = static_cast<float *>(PinnedPoolTake(bytes));
      std::memcpy(pinned_, rows, bytes);
      return;
    }
    if (ToDevice(rows)) return;
  }
  host_ = static_cast<float *>(HostPoolTake(bytes));
  ParallelFor(count, [&](size_t b, size_t e) { std::memcpy(host_ + b, rows + b, (e - b) * sizeof(float)); });
}

FloatRows::~FloatRows() {
  // (who reads the rows on the device waits for it before it returns)
  if (device_) g_device_bytes -= n_ * columns_ * sizeof(float);
  DevicePoolGive(device_);
  PinnedPoolGive(pinned_);
  HostPoolGive(host_);
}

bool FloatRows::ToDevice(const float *from) {
  const size_t bytes = n_ * columns_ * sizeof(float);
  if (bytes > kDeviceRowsBytes) return false;
  if ((g_device_bytes += bytes) > kAllDeviceRowsBytes) {
    g_device_bytes -= bytes;
    return false;
  }
  try {
    PooledStream stream;
    device_ = static_cast<float *>(DevicePoolTake(bytes));
    device_id_ = CurrentDevice();
    CopyToDevice(device_, from, bytes, stream.s);
    return true;
  } catch (const std::exception &) {  // no memory there: the rows stay on the host
    DevicePoolGive(device_);
    device_ = nullptr;
    g_device_bytes -= bytes;
    return false;
  }
}

const float *FloatRows::OnHost() {
  std::lock_guard<std::mutex> lock(mutex_);
  if (pinned_) return pinned_;
  if (!host_ && device_) {
    const size_t bytes = n_ * columns_ * sizeof(float);
    const OnDeviceOf device(device_id_);  // (the caller may use another one)
    PooledStream stream;
    float *p = static_cast<float *>(HostPoolTake(bytes));
    try {
      CopyToHost(p, device_, bytes, stream.s);
    } catch (...) {
      HostPoolGive(p);
      throw;
    }
    host_ = p;
  }
  return host_;
}

const float *FloatRows::OnDevice() {
  std::lock_guard<std::mutex> lock(mutex_);
  if (pinned_) return pinned_;
  if (device_) return device_id_ == CurrentDevice() ? device_ : nullptr;
  if (host_ && ToDevice(host_)) return device_;
  return nullptr;
}

}  // namespace arb
