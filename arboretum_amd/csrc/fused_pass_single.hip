#include "fused_pass_launch.h"

namespace arb {

template <bool WRITE>
static void Launch(bool group, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a) {
  if (hi) LaunchFused<false, WRITE, false, false, 1>(nq, st, grid, a);
  else if (!group) LaunchFused<false, WRITE, false, false>(nq, st, grid, a);
  else LaunchFused<false, WRITE, true, false>(nq, st, grid, a);
}

void LaunchFusedSingle(bool write, bool group, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a) {
  if (write) Launch<true>(group, hi, nq, st, grid, a);
  else Launch<false>(group, hi, nq, st, grid, a);
}

}  // namespace arb
