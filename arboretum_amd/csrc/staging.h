// Copies between ordinary host memory and the device through pinned blocks.
#ifndef ARBORETUM_AMD_STAGING_H_
#define ARBORETUM_AMD_STAGING_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

namespace arb {

// Host memory that is not pinned reaches the device through a few pinned blocks of kStageBytes:
// host threads fill or empty one while the copy engine works on another.  The runtime's own copy of
// pageable memory moves it on one thread (42 MB back to a fresh array: 8 ms, here 1.5).
constexpr size_t kStageBytes = (size_t)4 << 20;
constexpr int kStageSlots = 4;

// Blocks until `dst` holds the bytes (to the host) or `src` has been read (to the device; the copy
// itself is enqueued on `stream`, and later work on that stream finds the bytes).
void CopyToHost(void *dst, const void *src, size_t bytes, hipStream_t stream);
void CopyToDevice(void *dst, const void *src, size_t bytes, hipStream_t stream);

// The general form of the second: pieces of `bytes_of(k)` bytes, at most kStageBytes each, k = 0 ...
// pieces - 1, are filled by `fill(k, pinned)`, copied to `dst_of(k)`, and `then(k)` may enqueue work on
// that piece on the stream.  `fill` runs on the calling thread (it may use ParallelFor).
void StageToDevice(size_t pieces, const std::function<size_t(size_t)> &bytes_of,
                   const std::function<void(size_t, void *)> &fill, const std::function<void *(size_t)> &dst_of,
                   const std::function<void(size_t)> &then, hipStream_t stream);

}  // namespace arb
#endif  // ARBORETUM_AMD_STAGING_H_
