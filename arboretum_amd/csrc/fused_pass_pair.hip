#include "fused_pass_launch.h"

namespace arb {

template <bool WRITE>
static void Launch(bool group, bool pack, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a) {
  if (hi && pack) LaunchFused<true, WRITE, false, true, 1>(nq, st, grid, a);
  else if (hi) LaunchFused<true, WRITE, false, false, 1>(nq, st, grid, a);
  else if (pack && !group) LaunchFused<true, WRITE, false, true>(nq, st, grid, a);
  else if (pack) LaunchFused<true, WRITE, true, true>(nq, st, grid, a);
  else if (!group) LaunchFused<true, WRITE, false, false>(nq, st, grid, a);
  else LaunchFused<true, WRITE, true, false>(nq, st, grid, a);
}

void LaunchFusedPair(bool write, bool group, bool pack, bool hi, int nq, hipStream_t st, unsigned grid, const FusedArgs &a) {
  if (write) Launch<true>(group, pack, hi, nq, st, grid, a);
  else Launch<false>(group, pack, hi, nq, st, grid, a);
}

}  // namespace arb
