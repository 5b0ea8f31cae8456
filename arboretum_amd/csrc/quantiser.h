// Thresholds of feature columns by a device radix sort.
#ifndef ARBORETUM_AMD_QUANTISER_H_
#define ARBORETUM_AMD_QUANTISER_H_

#include <hip/hip_runtime.h>

#include <cstddef>

namespace arb {

// Work memory for `columns` columns of n values at a time (8 n bytes each, and little more).
struct SortWorkspace;
SortWorkspace *CreateSortWorkspace(size_t n, int hist_size, int columns);
void FreeSortWorkspace(SortWorkspace *ws);  // nothing that uses it may be pending

// Thresholds of `columns` columns (no more than the workspace is for) d_cols[columns][n]: d_thr gets
// hist_size floats per column (+INF where unset), d_sizes the number of real bins, d_has_nan
// whether a NaN is present.  Enqueued on `st`.
void DeviceThresholds(SortWorkspace *ws, const float *d_cols, int columns, float *d_thr, int *d_sizes,
                      unsigned *d_has_nan, hipStream_t st);

// Columns [f0, f0 + nf) of n row-major rows of F floats -> d_cols[column * ld + at + row].
void RowsToColumns(const float *d_rows, size_t n, int F, int f0, int nf, float *d_cols, size_t ld, size_t at,
                   hipStream_t st);

}  // namespace arb
#endif  // ARBORETUM_AMD_QUANTISER_H_
