// The feature values of a float matrix, row-major as they were handed in.
#ifndef ARBORETUM_AMD_FLOAT_ROWS_H_
#define ARBORETUM_AMD_FLOAT_ROWS_H_

#include <cstddef>
#include <mutex>

namespace arb {

// Where the rows are kept.  Everything but the host walk and the exact method's sort reads them on the
// GPU, so in a process that uses the GPU they go straight there, through pinned blocks, and host
// memory never holds a copy.
//   - up to kPinnedRowsBytes: one pinned block, which kernels read where it is (a copy to the device
//     costs more than its bytes);
//   - up to kDeviceRowsBytes, and kAllDeviceRowsBytes over all matrices: device memory;
//   - more, no memory there, or no GPU in use by this process yet: host memory, and on the device from
//     the first OnDevice() on if they fit there (a process that only builds matrices never starts
//     the GPU, and may fork).
// Rows on the device are memory of their matrix: they stay until it is freed, and a streamed matrix keeps
// that much less of its bins resident meanwhile (its own rows never matter: where they fit, its bins, a quarter
// of their size, do).
class FloatRows {
 public:
  FloatRows(const float *rows, size_t n, size_t columns);
  ~FloatRows();
  FloatRows(const FloatRows &) = delete;
  FloatRows &operator=(const FloatRows &) = delete;

  // [n][columns] on the host; rows that are only on the device are fetched once.
  const float *OnHost();
  // [n][columns] for kernels on the current device, complete for every stream; null when they do not
  // fit there or are on another device.
  const float *OnDevice();

 private:
  bool ToDevice(const float *from);
  const size_t n_, columns_;
  std::mutex mutex_;
  float *host_ = nullptr, *pinned_ = nullptr, *device_ = nullptr;
  int device_id_ = 0;
};

}  // namespace arb
#endif  // ARBORETUM_AMD_FLOAT_ROWS_H_
