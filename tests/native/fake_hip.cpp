#include "fake_hip.h"

#include <cstdlib>
#include <cstring>

namespace fake {
thread_local int current = 0;
size_t capacity = (size_t)1 << 40;
std::mutex mutex;
std::map<void *, std::pair<int, size_t>> blocks;
std::map<void *, size_t> pinned;
std::map<hipStream_t, int> streams;
size_t BytesOn(int device) {
  size_t n = 0;
  for (const auto &b : blocks)
    if (b.second.first == device) n += b.second.second;
  return n;
}
}  // namespace fake

extern "C" {
hipError_t hipGetDevice(int *device) {
  *device = fake::current;
  return hipSuccess;
}
hipError_t hipSetDevice(int device) {
  fake::current = device;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  if (fake::BytesOn(fake::current) + bytes > fake::capacity) return hipErrorOutOfMemory;
  *p = std::malloc(bytes);
  fake::blocks[*p] = {fake::current, bytes};
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  if (!fake::blocks.erase(p)) std::abort();
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  *p = std::malloc(bytes);
  fake::pinned[*p] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  if (!fake::pinned.erase(p)) std::abort();
  std::free(p);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  *s = static_cast<hipStream_t>(std::malloc(1));
  fake::streams[*s] = fake::current;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::lock_guard<std::mutex> lock(fake::mutex);
  if (!fake::streams.erase(s)) std::abort();
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// at once, in order; a copy that touches memory of another device than its stream's is refused
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t s) {
  {
    std::lock_guard<std::mutex> lock(fake::mutex);
    for (const auto &b : fake::blocks)
      for (const void *p : {(const void *)to, from})
        if (p >= b.first && p < static_cast<char *>(b.first) + b.second.second && fake::streams.at(s) != b.second.first)
          return hipErrorInvalidDevice;
  }
  std::memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "an error"; }
}
