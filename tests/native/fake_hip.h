// Some calls of the HIP runtime over host memory, with as many devices as a test asks for: the pools are
// checked on machines without a GPU, and with several.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <map>
#include <mutex>

namespace fake {
extern thread_local int current;                    // hipSetDevice
extern size_t capacity;                             // bytes of a device; hipMalloc beyond it fails
extern std::mutex mutex;                            // guards what follows
extern std::map<void *, std::pair<int, size_t>> blocks;   // device blocks in existence: device, bytes
extern std::map<void *, size_t> pinned;
extern std::map<hipStream_t, int> streams;          // streams in existence: device
size_t BytesOn(int device);
}  // namespace fake
