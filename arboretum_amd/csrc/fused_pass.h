// Launches of the fused partition + histogram pass (k_part_hist); its many instances are compiled in
// two files of their own.
#ifndef ARBORETUM_AMD_FUSED_PASS_H_
#define ARBORETUM_AMD_FUSED_PASS_H_
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "kernels_split.h"

namespace arb {

struct FusedArgs {
  const uint32_t *bins;
  uint32_t *bins_out;
  size_t stride;
  int F;
  const float *g;
  float *g_out;
  const float *h;
  float *h_out;
  const int *shifts;
  const SplitRec *split;
  const NodeSum *tot;
  const unsigned *seg_start;
  const WorkItem *work;
  const unsigned *n_work;
  unsigned *cursor;     // claims destinations (null: read item_base)
  unsigned *item_base;  // claimed destination bases, two per work item
  unsigned long long *slab;
  int slab_entries;
  const uint32_t *split_bins;  // start of the whole matrix
  int q0;                      // first quad of this launch
  unsigned rows_per_item;      // most rows of a work item
  LevelScan scan;              // cand set: the pass finds the splits of its parents itself
};

// with hessians (pack: packed logistic gradients) / without.  write: the rows move to the children
// order; group: one group of quads of a wider matrix; hi: rows with a ninth-bit word; nq: quads.
void LaunchFusedPair(bool write, bool group, bool pack, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a);
void LaunchFusedSingle(bool write, bool group, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a);

}  // namespace arb
#endif  // ARBORETUM_AMD_FUSED_PASS_H_
