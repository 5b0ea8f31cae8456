// The choice of the instance of k_part_hist, shared by the two files that compile them.
#ifndef ARBORETUM_AMD_FUSED_PASS_LAUNCH_H_
#define ARBORETUM_AMD_FUSED_PASS_LAUNCH_H_
#include "fused_pass.h"
#include "kernels_launch.h"
#include "kernels_partition.h"

namespace arb {
namespace {

template <bool PAIR, int NQ, bool WRITE, bool GROUP, bool PACK, int HI>
void LaunchFusedNQ(hipStream_t st, unsigned grid, const FusedArgs &a) {
  const size_t lds = HistLdsBytes(NQ, PAIR, HI != 0);
#define ARB_FUSED(KERNEL)                                                                                             \
  do {                                                                                                                \
    static std::once_flag configured;                                                                                 \
    AllowLdsOnce(configured, KERNEL<PAIR, NQ, WRITE, GROUP, PACK, HI>, lds);                                          \
    hipLaunchKernelGGL((KERNEL<PAIR, NQ, WRITE, GROUP, PACK, HI>), dim3(grid), dim3(kHistThreads), lds, st,           \
                       a.bins + (size_t)a.q0 * a.stride, a.bins_out ? a.bins_out + (size_t)a.q0 * a.stride : nullptr, \
                       a.stride, a.F, a.g, a.g_out, a.h, a.h_out, a.shifts, a.split, a.tot, a.seg_start, a.work,      \
                       a.n_work, a.cursor, a.item_base, a.slab, a.slab_entries, a.split_bins, a.q0, a.scan);          \
  } while (0)
  // one chunk of rows per wave; the last level, which moves none, is as fast in half-empty waves up to half of that
  // (300,000 rows x 29, items of 2048: 12.4 us by k_part_hist, 13.1; 10,000 x 28, items of 1024: 8.4, 8.0)
  const bool small = a.rows_per_item <= (WRITE ? kChunkStep : kChunkStep / 2);
  if (small && (GROUP || a.scan.cand != nullptr)) ARB_FUSED(k_part_hist_small);
  else ARB_FUSED(k_part_hist);
#undef ARB_FUSED
}

template <bool PAIR, bool WRITE, bool GROUP, bool PACK, int HI = 0>
void LaunchFused(int nq, hipStream_t st, unsigned grid, const FusedArgs &a) {
#define ARB_CASE(N) \
  case N: LaunchFusedNQ<PAIR, N, WRITE, GROUP, PACK, HI>(st, grid, a); break;
  switch (nq) {
    ARB_CASE(1) ARB_CASE(2) ARB_CASE(3) ARB_CASE(4) ARB_CASE(5) ARB_CASE(6) ARB_CASE(7) ARB_CASE(8)
    default: throw std::runtime_error("internal: bad quad count");
  }
#undef ARB_CASE
}

}  // namespace
}  // namespace arb
#endif  // ARBORETUM_AMD_FUSED_PASS_LAUNCH_H_
