// The exact method's scan looks only at places whose ExSides comes near the largest of the wave: the place it
// picks is the one that looking at all of them picks, over random nodes of every kind of sums.
#include <cfloat>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../arboretum_amd/csrc/exact_filter.h"

using namespace arb;

struct Node {
  std::vector<long long> g, h;  // running sums, fixed point
  long long gt = 0, ht = 0;
  int sg = 0, sh = 0;
  GainParams p{};
};

typedef std::mt19937_64 Rng;
static double Uniform(Rng &r) { return std::uniform_real_distribution<double>(0, 1)(r); }

// kind: what is special about the node
static Node Make(Rng &rng, bool pair, int kind) {
  Node n;
  const size_t places = 2 + rng() % 200;
  const double scale = kind == 1 ? std::ldexp(1.0, (int)(rng() % 160) - 80) : 1.0;
  n.sg = FixShiftFromMax((float)scale);
  n.sh = 32;
  const bool ties = rng() % 2;  // sums that hardly change from place to place: gains next to each other
  for (size_t i = 0; i < places; ++i) {
    double g = (Uniform(rng) - 0.5) * scale, h = Uniform(rng) * 0.25;
    if (ties && i > 0 && i + 1 < places) g = kind == 1 ? 0.0 : g * 1e-7, h *= 1e-7;
    if (kind == 2) h *= 1e-6;  // tiny hessians
    n.gt += kind == 3 ? (long long)(g * (1 << 30)) : ToFixed((float)g, n.sg);
    n.ht += kind == 3 ? (long long)(h * 0x1p32) : ToFixed((float)h, n.sh);
    n.g.push_back(n.gt);
    n.h.push_back(n.ht);
  }
  n.p.min_leaf_size = rng() % 3 == 0 ? (unsigned)(rng() % 5) : 0u;
  n.p.min_child_weight = rng() % 3 == 0 ? (float)Uniform(rng) : 0.0f;
  n.p.gamma_absolute = rng() % 4 == 0 ? (float)(Uniform(rng) * scale * scale) : 0.0f;
  n.p.gamma_relative = rng() % 4 == 0 ? (float)(Uniform(rng) * 0.1) : 0.0f;
  n.p.lambda = rng() % 3 == 0 ? 0.0f : rng() % 2 ? 1.0f : (float)(Uniform(rng) * 10);
  if (kind == 1 && rng() % 3 == 0) n.p.lambda = std::ldexp(1.0f, -(int)(rng() % 100));
  if (kind == 2 && rng() % 2 == 0) n.p.lambda = 1e-10f;
  if (kind == 3) {
    // hessians and lambda of about 2^62: the product of the denominators is about 2^126, where its reciprocal
    // stops being a normal float
    n.p.lambda = std::ldexp(1.0f, 61 + (int)(rng() % 2));
    n.sh = -22 - (int)(rng() % 8);
    n.sg = 0;
  }
  return n;
}

// The best place (the last of equal ones), and its gain; `look`: which are looked at.
template <bool PAIR, bool F64>
static int Pick(const Node &n, const std::vector<bool> &look, float *gain) {
  const double gt = FromFixed<F64>(n.gt, n.sg), ht = PAIR ? FromFixed<F64>(n.ht, n.sh) : 0.0;
  const float parent = ExParentGain<PAIR, F64>(gt, ht, n.g.size(), n.p);
  int best = -1;
  *gain = 0.0f;
  for (size_t i = 0; i + 1 < n.g.size(); ++i) {
    if (!look[i]) continue;
    const double gl = FromFixed<F64>(n.g[i], n.sg), hl = PAIR ? FromFixed<F64>(n.h[i], n.sh) : 0.0;
    const float g = ExSplitGain<PAIR, F64>(gl, hl, i + 1, gt, ht, n.g.size(), n.p, parent);
    const float same = SplitGain<PAIR, F64>(gl, hl, i + 1, gt, ht, n.g.size(), n.p);
    if (std::memcmp(&g, &same, 4) != 0) {
      std::printf("ExSplitGain is not SplitGain\n");
      std::exit(1);
    }
    if (g > 0.0f && g >= *gain) {
      *gain = g;
      best = (int)i;
    }
  }
  return best;
}

// v_rcp_f32: within one unit in the last place (`off`), results below the normal floats flushed to zero
static float Rcp(float x, int off) {
  float r = 1.0f / x;
  if (off > 0) r = std::nextafterf(r, INFINITY);
  if (off < 0) r = std::nextafterf(r, 0.0f);
  return std::fabs(r) < FLT_MIN ? 0.0f : r;
}

struct Counts {
  long nodes = 0, wrong = 0, places = 0, looked = 0, pruned = 0;
};

template <bool PAIR, bool F64>
static void Check(Rng &rng, int kind, float margin, Counts *c) {
  const Node n = Make(rng, PAIR, kind);
  const size_t m = n.g.size();
  const double gt = FromFixed<F64>(n.gt, n.sg), ht = PAIR ? FromFixed<F64>(n.ht, n.sh) : 0.0;
  std::vector<float> sides(m, INFINITY);
  float most = 0.0f;
  const bool prune = ExPrunes<PAIR>(ht, m, n.p);
  c->pruned += prune;
  for (size_t i = 0; prune && i + 1 < m; ++i) {
    const int off = (int)(rng() % 3) - 1;
    sides[i] = ExSides<PAIR, F64>(FromFixed<F64>(n.g[i], n.sg), PAIR ? FromFixed<F64>(n.h[i], n.sh) : 0.0, i + 1, gt, ht, m,
                                  n.p, [off](float x) { return Rcp(x, off); });
    if (sides[i] <= kExMostSides) most = std::fmax(most, sides[i]);
  }
  const float least = !prune ? 0.0f : ExLeastSides<PAIR>(most, margin);
  std::vector<bool> look(m), all(m, true);
  for (size_t i = 0; i < m; ++i) look[i] = !(sides[i] < least);
  float ga, gb;
  const int a = Pick<PAIR, F64>(n, all, &ga), b = Pick<PAIR, F64>(n, look, &gb);
  ++c->nodes;
  c->places += (long)m;
  for (size_t i = 0; i + 1 < m; ++i) c->looked += look[i];
  if (a != b || ga != gb) ++c->wrong;
}

int main(int argc, char **argv) {
  const int kind = std::atoi(argv[1]);
  const long nodes = std::atol(argv[2]);
  const float margin = argc > 3 ? (float)std::atof(argv[3]) : kExMargin;
  Rng rng(kind + 1);
  Counts c;
  for (long i = 0; i < nodes; ++i) {
    Check<false, false>(rng, kind, margin, &c);
    Check<false, true>(rng, kind, margin, &c);
    Check<true, false>(rng, kind, margin, &c);
    Check<true, true>(rng, kind, margin, &c);
  }
  std::printf("%ld %ld %ld %ld %ld\n", c.nodes, c.wrong, c.places, c.looked, c.pruned);
  return 0;
}
