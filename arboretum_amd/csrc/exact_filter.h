// The gains of the exact method's scan: at which places of a list they have to be computed at all, and how.
// Host and device: the CPU tests compile this header.
#ifndef ARBORETUM_AMD_EXACT_FILTER_H_
#define ARBORETUM_AMD_EXACT_FILTER_H_
#include <cmath>

#include "gain.h"

namespace arb {

// SplitGain (gain.h) with the parent's term, which is the same at every place of a node, taken
// from the caller: `parent` = SideGain of the node's totals at their leaf weight.  The same
// operations in the same order, so the same bits.
template <bool PAIR, bool F64>
ARB_HD float ExParentGain(double gt, double ht, unsigned long long ct, const GainParams &p) {
  return SideGain<PAIR, F64>(gt, ht, ct, LeafWeight<PAIR, F64>(gt, ht, ct, p), p);
}
template <bool PAIR, bool F64>
ARB_HD float ExSplitGain(double gl, double hl, unsigned long long cl, double gt, double ht,
                         unsigned long long ct, const GainParams &p, float parent) {
  const unsigned long long cr = ct - cl;
  double gr, hr;
  if (F64) {
    gr = gt - gl;
    hr = ht - hl;
  } else {
    gr = (double)((float)gt - (float)gl);
    hr = (double)((float)ht - (float)hl);
  }
  if (cl < p.min_leaf_size || cr < p.min_leaf_size) return 0.0f;
  if (PAIR) {
    if (F64) {
      if (!(fabs(hl) >= (double)p.min_child_weight && fabs(hr) >= (double)p.min_child_weight)) return 0.0f;
    } else {
      if (!(fabsf((float)hl) >= p.min_child_weight && fabsf((float)hr) >= p.min_child_weight)) return 0.0f;
    }
  }
  const float l = SideGain<PAIR, F64>(gl, hl, cl, LeafWeight<PAIR, F64>(gl, hl, cl, p), p);
  const float r = SideGain<PAIR, F64>(gr, hr, cr, LeafWeight<PAIR, F64>(gr, hr, cr, p), p);
  const float diff = l + r - parent;
  return (float)(diff > p.gamma_absolute && diff > p.gamma_relative * parent) * diff;
}

// ---- which places can be the best of a wave's
// ExSides is the sum of the two sides' gains at a place, S = g_l^2 / d_l + g_r^2 / d_r (g the gradients of a side,
// d its hessians, or rows, + lambda): ExSplitGain but for the parent's term, in a sixth of its instructions (single
// precision, no division).  Only places whose ExSides is within kExMargin of the wave's largest are looked at
// (ExSplitGain); the others cannot be the best, nor tie with it.  Why, with e = 2^-24:
//   ExSides is within 5 e of S: numerator and denominator are double, rounded once each (e, e), the reciprocal is within one
//     unit in the last place (2 e), the product is rounded (e); as long as none of them leaves the normal floats (below).
//   fl(l + r) of ExSplitGain is within 5 e of S.  A side is 2 g w - d w^2 at w = (g / d) (1 + a): g^2 / d (1 - a^2),
//     so the rounding of w does not count; in single precision g w is rounded (2 e: it stands twice) and so is d (e); the
//     side is rounded (e) and so is the sum of the two (e).
//   A place with ExSides < (1 - m) times the largest has S < S_max (1 + 10 e) (1 - m), so its fl(l + r) is less than
//     that of the largest by (m - 20 e) S_max and more: 2.8e-6 S_max for m = 4e-6.
//   The parent's term is between 0 and S (g^2 / d is convex, lambda >= 0), so the difference l + r - parent is rounded by
//     e S_max at most, and stays less than the largest one.  The limits gamma are the same for both.
constexpr float kExMargin = 4e-6f;
constexpr float kExMostSides = 3.0e38f;  // larger (or not a number): not a maximum, and looked at

// Whether the places of a node of the sums (., ht, ct) are left out by that rule at all; else every one is looked at.
//   No alpha and no bound on the weights: those make the gain another function.
//   The denominators stay where floats and their reciprocals are normal (v_rcp_f32 gives zero past 2^126).  Hessians are not
//     negative and multiples of 2^-32, so a side that has any has a d of 2^-32 or lambda at least: d_l d_r is between
//     1e-20 and (ht + lambda)^2.
template <bool PAIR>
ARB_HD bool ExPrunes(double ht, unsigned long long ct, const GainParams &p) {
  const double most = (PAIR ? ht : (double)ct) + (double)p.lambda;
  return p.alpha == 0.0f && p.max_leaf_weight == 0.0f && most * most <= 1e37 && (p.lambda == 0.0f || p.lambda >= 1e-10f);
}

// The least ExSides of a place worth a look.  A numerator below 1e-37 loses digits, and so does a product: they are less than
// 1e-17 of gain (PAIR; 1e-37 with rows for hessians, d_l d_r >= 1), so nothing is left out next to gains of that size.
template <bool PAIR>
ARB_HD float ExLeastSides(float most, float margin = kExMargin) {
  return most < (PAIR ? 1e-10f : 1e-30f) ? 0.0f : most * (1.0f - margin);
}

// rcp: 1 / x within one unit in the last place.  Negative for a place that has no gain by the limits on leaves, infinite or
// not a number for one to be looked at in any case.
template <bool PAIR, bool F64, typename Rcp>
ARB_HD float ExSides(double gl, double hl, unsigned long long cl, double gt, double ht, unsigned long long ct,
                     const GainParams &p, Rcp rcp) {
  const unsigned long long cr = ct - cl;
  const double gr = F64 ? gt - gl : (double)((float)gt - (float)gl);
  double hr = F64 ? ht - hl : (double)((float)ht - (float)hl);
  bool none = cl < p.min_leaf_size || cr < p.min_leaf_size;
  if (PAIR) none = none || !(fabs(hl) >= (double)p.min_child_weight && fabs(hr) >= (double)p.min_child_weight);
  if (!PAIR) {
    hl = (double)(float)cl;
    hr = (double)(float)cr;
  }
  const double dl = hl + (double)p.lambda, dr = hr + (double)p.lambda;
  const float v = (float)(gl * gl * dr + gr * gr * dl) * rcp((float)(dl * dr));
  // (LeafWeight: such a side has the weight 0)
  const bool zero = !(hl >= (double)p.min_child_weight && hr >= (double)p.min_child_weight) || !(dl > 0.0 && dr > 0.0);
  return none ? -1.0f : zero ? INFINITY : v;
}

}  // namespace arb
#endif  // ARBORETUM_AMD_EXACT_FILTER_H_
