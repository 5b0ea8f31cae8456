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
  static std::once_flag configured;
  AllowLdsOnce(configured, k_part_hist<PAIR, NQ, WRITE, GROUP, PACK, HI>, lds);
  hipLaunchKernelGGL((k_part_hist<PAIR, NQ, WRITE, GROUP, PACK, HI>), dim3(grid), dim3(kHistThreads), lds, st,
                     a.bins + (size_t)a.q0 * a.stride, a.bins_out ? a.bins_out + (size_t)a.q0 * a.stride : nullptr,
                     a.stride, a.F, a.g, a.g_out, a.h, a.h_out, a.shifts, a.split, a.tot, a.seg_start, a.work,
                     a.n_work, a.cursor, a.item_base, a.slab, a.slab_entries, a.split_bins, a.q0, a.scan);
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
