// Exact method over sorted row lists: features with more distinct values than a histogram holds.
//
// Every feature keeps the rows of every node of the current level as one list of row ids in
// ascending order of the feature's value (the reference sorts every column once and keeps the
// node segments sorted, src/core/continuous_tree_grower.cu).  Per level and feature: the running
// sums of the gradients along the list give, at every place where the value changes, the
// candidate "values up to here go left"; the best one per (node, feature) goes to the same
// selection as the histogram method's candidates, and a stable partition by the selected splits
// turns the lists of the parents into the lists of the children.
//
// The candidates are those of a histogram with one slot per distinct value (rank): a slot that
// is empty in a node has the gain of the slot before it, and ties go to the highest slot
// (builder.h:39-49), so the candidate between two neighbouring values of a node is the slot just
// below the upper one, and its threshold is that upper value: the smallest value that goes right.
#ifndef ARBORETUM_AMD_KERNELS_EXACT_H_
#define ARBORETUM_AMD_KERNELS_EXACT_H_
#include "device_common.h"
#include "exact_filter.h"
#include "gain.h"
#include "kernels_split.h"

namespace arb {
namespace {

constexpr int kExThreads = 256;
constexpr int kExPer = 8;                          // list places per thread
constexpr unsigned kExItem = kExThreads * kExPer;  // list places per work item

struct ExSum {
  long long g, h;
};
__device__ __forceinline__ ExSum operator+(const ExSum &a, const ExSum &b) { return ExSum{a.g + b.g, a.h + b.h}; }
__device__ __forceinline__ ExSum ExShflUp(const ExSum &v, int off) {
  return ExSum{__shfl_up(v.g, off), __shfl_up(v.h, off)};
}
__device__ __forceinline__ unsigned ExShflUp(unsigned v, int off) { return __shfl_up(v, off); }
__device__ __forceinline__ ExSum ExZero(const ExSum *) { return ExSum{0, 0}; }
__device__ __forceinline__ unsigned ExZero(const unsigned *) { return 0u; }

// Inclusive scan over the workgroup's threads (kExThreads of them) of one value per thread;
// *total: the sum over all threads.  s_wave: kExThreads / 64 entries.
template <typename T>
__device__ __forceinline__ T ExBlockScan(T v, T *s_wave, T *total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int off = 1; off < 64; off <<= 1) {
    const T o = ExShflUp(v, off);
    if (lane >= off) v = v + o;
  }
  __syncthreads();  // s_wave may still be read from a scan before
  if (lane == 63) s_wave[wave] = v;
  __syncthreads();
  T before = ExZero((const T *)nullptr), all = ExZero((const T *)nullptr);
  for (int w = 0; w < kExThreads / 64; ++w) {
    if (w < wave) before = before + s_wave[w];
    all = all + s_wave[w];
  }
  *total = all;
  return before + v;
}

// The lists of a level: for every feature the rows of every node in ascending order of the
// feature's value, and next to each row id what the passes need of that row, so that they read
// it in list order instead of gathering it by row: the row's rank in this feature and its
// gradients (the root's ids and ranks are the same for every tree; its gradients are gathered
// once per tree, k_ex_gather).
struct ExLists {
  const unsigned *ids;    // [F][stride]
  const unsigned *ranks;  // [F][stride]
  const float *g, *h;     // [F][stride]; h null without hessians
};

// Eight consecutive words of a list from place p0, `fill` past `end`.
template <typename T>
__device__ __forceinline__ void ExLoad8(const T *__restrict__ base, unsigned p0, unsigned end, T fill, T *out) {
  static_assert(sizeof(T) == 4, "lists hold 32-bit words");
  if ((p0 & 3u) == 0 && p0 + kExPer <= end) {
    const uint4 a = *reinterpret_cast<const uint4 *>(base + p0);
    const uint4 b = *reinterpret_cast<const uint4 *>(base + p0 + 4);
    const unsigned w[kExPer] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < kExPer; ++j) __builtin_memcpy(&out[j], &w[j], 4);
  } else {
#pragma unroll
    for (int j = 0; j < kExPer; ++j) out[j] = p0 + j < end ? base[p0 + j] : fill;
  }
}

// The fixed-point gradients (at most 2^30 in magnitude) of the rows at the places [p0, p0 + kExPer) of
// feature f's list, zero past `end`.
// PACK: one float per row holds both (logistic gradients of 0/1 labels, PackGrad); no h lists.
template <bool PAIR, bool PACK>
__device__ __forceinline__ void ExLoadGrads(const ExLists &ls, size_t fbase, unsigned p0, unsigned end, int sg, int sh,
                                            int *g, int *h) {
  float gv[kExPer], hv[kExPer];
  ExLoad8(ls.g + fbase, p0, end, 0.0f, gv);
  if (PAIR && !PACK) ExLoad8(ls.h + fbase, p0, end, 0.0f, hv);
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    float g1 = gv[j], h1 = PAIR && !PACK ? hv[j] : 0.0f;
    if (PACK) UnpackGrad(gv[j], &g1, &h1);
    g[j] = p0 + j < end ? (int)ToFixed(g1, sg) : 0;
    h[j] = PAIR && p0 + j < end ? (int)ToFixed(h1, sh) : 0;
  }
}

// Sums of N values over the workgroup (kExThreads threads), valid in every thread.
template <int N>
__device__ __forceinline__ void ExBlockSums(long long (&v)[N], long long (*s_wave)[N]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = WaveSumLL(v[k]);
  __syncthreads();  // s_wave may still be read from a sum before
  if (lane == 0)
    for (int k = 0; k < N; ++k) s_wave[wave][k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    v[k] = 0;
    for (int w = 0; w < kExThreads / 64; ++w) v[k] += s_wave[w][k];
  }
}

// The work plan of a level and, per feature and work item, the sum of the gradients over that piece of the
// feature's list: made by the pass that writes the lists (k_ex_gather, k_ex_scatter).
struct ExPlan {
  WorkItem *work;
  unsigned *n_work, *node_first, *node_items;
  ExSum *part;  // [F][max_items]
};
// Up to this many work items in the matrix a workgroup adds up what it needs of the items before its own; more,
// and k_ex_offsets does it for all.  (400,000 rows are 196 items: a few of them per thread at most, and a launch
// of 4.6 us less, twice a level.)
constexpr unsigned kExFoldItems = 512;

// Up to this many pieces of lists (work items x features) the scan filters its places.  Levels 0, 1 and 7 with / without, us, 28
// features: 400,000 rows (5500) 65, 67, 77 / 74, 66, 84; 1 M (14,000) 163, 170, 160 / 181, 163, 172; 3 M (41,000) 389, 479, 408 /
// 392, 394, 406; 10.5 M (144,000) 1500, 1829, 1516 / 1432, 1435, 1376.
constexpr size_t kExFilterItems = 16384;

// grid (L, F), one wave: exclusive scan of `part` over the work items of every node, per feature.
template <typename T>
__global__ void __launch_bounds__(64)
k_ex_offsets(const T *__restrict__ part, T *__restrict__ off, const unsigned *__restrict__ node_first,
             const unsigned *__restrict__ node_items, unsigned max_items) {
  const unsigned nd = blockIdx.x, f = blockIdx.y, lane = threadIdx.x;
  const unsigned first = node_first[nd];
  unsigned cnt = node_items[nd];
  if (cnt == 0xffffffffu) cnt = 0;
  T carry = ExZero((const T *)nullptr);
  for (unsigned base = 0; base < cnt; base += 64) {
    const unsigned k = base + lane;
    const T own = k < cnt ? part[(size_t)f * max_items + first + k] : ExZero((const T *)nullptr);
    T v = own;
    for (int o = 1; o < 64; o <<= 1) {
      const T up = ExShflUp(v, o);
      if ((int)lane >= o) v = v + up;
    }
    // exclusive: the sum of the items before this one
    T excl = carry;
    {
      const T prev = ExShflUp(v, 1);
      if (lane > 0) excl = excl + prev;
    }
    if (k < cnt) off[(size_t)f * max_items + first + k] = excl;
    T last;
    if constexpr (sizeof(T) == sizeof(unsigned)) {
      last = __shfl(v, 63);
    } else {
      last = ExSum{__shfl(v.g, 63), __shfl(v.h, 63)};
    }
    carry = carry + last;
  }
}

__device__ __forceinline__ bool ExBetter(float og, int ob, float gain, int bin) {
  return ob >= 0 && (bin < 0 || og > gain || (og == gain && ob > bin));
}

// grid (items, F): running sums along every work item's piece of every list (on top of `off`, the
// sums of the node's items before it), the gain wherever the rank changes to the next place of the
// node, and the best candidate of the piece, ties to the highest rank.
// best: [F][max_items].
// What bounds it: the gains in double precision (21 of 50 us a level at 400,000 rows x 20), then the latency of a
// chain of loads, scan and barriers, hidden by the workgroups of a CU.  Only the best place of a wave counts, so with
// FILTER the gains are computed where ExSides comes near the wave's largest (ExLeastSides): usually at one place or
// two of 512 (43 us; with fewer registers, six waves per SIMD, they spill: 76).  That shortens a workgroup, and costs
// arithmetic and registers that a chip full of workgroups has better use for (kExFilterItems).
template <bool PAIR, bool F64, bool PACK, bool FILTER>
__global__ void __launch_bounds__(kExThreads)
k_ex_scan(const ExLists ls, size_t stride, const int *__restrict__ shifts,
          const ExPlan plan, const ExSum *__restrict__ off, int root,
          NodeSum *tot, const unsigned *__restrict__ seg_start, GainParams gp,
          Cand *__restrict__ best, unsigned max_items) {
  __shared__ ExSum s_wave[kExThreads / 64];
  __shared__ Cand s_best[kExThreads / 64];
  const unsigned w = blockIdx.x, f = blockIdx.y;
  if (w >= *plan.n_work) return;
  const WorkItem it = plan.work[w];
  NodeSum t = tot[it.node];
  const unsigned node_start = seg_start[it.node], node_end = node_start + (unsigned)t.c;
  const size_t fbase = (size_t)f * stride;
  const int sg = shifts[0], sh = shifts[1];
  const unsigned p0 = it.begin + threadIdx.x * kExPer;
  int gq[kExPer], hq[kExPer];
  ExLoadGrads<PAIR, PACK>(ls, fbase, p0, it.end, sg, sh, gq, hq);
  // ranks at this thread's places and at the one after them (which may lie in the next item)
  unsigned rk[kExPer + 1];
  ExLoad8(ls.ranks + fbase, p0, node_end, 0u, rk);
  rk[kExPer] = p0 + kExPer < node_end ? ls.ranks[fbase + p0 + kExPer] : 0u;
  ExSum base{0, 0};
  if (off != nullptr) {  // uniform
    base = off[(size_t)f * max_items + w];
  } else {
    // The items of the node before this one; at the root also all of them, which are the root's totals.  Every
    // wave makes the sums for itself: no barrier, and the loads are under way with those of the lists.
    const unsigned end = root ? *plan.n_work : w, lane = threadIdx.x & 63;
    ExSum all{0, 0};
    for (unsigned k = it.first + lane; k < end; k += 64) {
      const ExSum x = plan.part[(size_t)f * max_items + k];
      if (k < w) base = base + x;
      all = all + x;
    }
    base = ExSum{__shfl(WaveSumLL(base.g), 0), PAIR ? __shfl(WaveSumLL(base.h), 0) : 0};
    if (root) {
      t.g = __shfl(WaveSumLL(all.g), 0);
      t.h = PAIR ? __shfl(WaveSumLL(all.h), 0) : 0;
      if (w == 0 && f == 0 && threadIdx.x == 0) tot[0] = t;
    }
  }
  ExSum own{0, 0};
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    own.g += gq[j];
    if (PAIR) own.h += hq[j];
  }
  ExSum total;
  const ExSum incl = ExBlockScan(own, s_wave, &total);
  long long lg = base.g + incl.g - own.g, lh = base.h + incl.h - own.h;

  Cand mine;
  mine.gain = 0.0f;
  mine.bin = -1;
  mine.left.g = mine.left.h = 0;
  mine.left.c = 0;
  const double GT = FromFixed<F64>(t.g, sg);
  const double HT = PAIR ? FromFixed<F64>(t.h, sh) : 0.0;
  const float parent = ExParentGain<PAIR, F64>(GT, HT, t.c, gp);
  const bool prune = FILTER && ExPrunes<PAIR>(HT, t.c, gp);
  // the places worth a look: bit j
  unsigned look = 0;
  float sides[kExPer], most = 0.0f;
  long long g_at = lg, h_at = lh;
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    const unsigned p = p0 + j;
    g_at += gq[j];
    if (PAIR) h_at += hq[j];
    sides[j] = INFINITY;
    if (p < it.end && p + 1 < node_end && rk[j] != rk[j + 1]) look |= 1u << j;
    if (prune)  // uniform
      sides[j] = ExSides<PAIR, F64>(FromFixed<F64>(g_at, sg), PAIR ? FromFixed<F64>(h_at, sh) : 0.0, p - node_start + 1, GT,
                                    HT, t.c, gp, [](float x) { return __builtin_amdgcn_rcpf(x); });
    if (((look >> j) & 1u) && sides[j] <= kExMostSides) most = fmaxf(most, sides[j]);
  }
  if (prune) {
    for (int o = 32; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o));
    const float least = ExLeastSides<PAIR>(most);
#pragma unroll
    for (int j = 0; j < kExPer; ++j)
      if (sides[j] < least) look &= ~(1u << j);  // (not finite: looked at)
  }
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    lg += gq[j];
    if (PAIR) lh += hq[j];
    const bool on = (look >> j) & 1u;
    if (__ballot(on) == 0ull) continue;  // uniform
    const unsigned long long lc = p0 + j - node_start + 1;
    float gn = 0.0f;
    if (on)
      gn = ExSplitGain<PAIR, F64>(FromFixed<F64>(lg, sg), PAIR ? FromFixed<F64>(lh, sh) : 0.0, lc, GT, HT, t.c, gp, parent);
    if (gn > 0.0f && gn >= mine.gain) {
      mine.gain = gn;
      mine.bin = (int)(rk[j + 1] - 1u);
      mine.left.g = lg;
      mine.left.h = lh;
      mine.left.c = lc;
    }
  }
  // highest gain, ties to the highest rank: one key, then the winner's sums
  const unsigned long long key = mine.bin < 0 ? 0ull : ((unsigned long long)__float_as_uint(mine.gain) << 32) | (unsigned)(mine.bin + 1);
  unsigned long long top = key;
  for (int o = 32; o > 0; o >>= 1) top = max(top, (unsigned long long)__shfl_xor(top, o));
  const int from = __ffsll((unsigned long long)__ballot(key == top)) - 1;  // (ranks of the places differ)
  if ((int)(threadIdx.x & 63) == from) s_best[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (threadIdx.x == 0) {
    mine = s_best[0];
    for (int k = 1; k < kExThreads / 64; ++k)
      if (ExBetter(s_best[k].gain, s_best[k].bin, mine.gain, mine.bin)) mine = s_best[k];
    best[(size_t)f * max_items + w] = mine;
  }
}

// Split of every node: the best candidate of its work items per feature (ties to the highest rank), the best
// feature of those active at the level (ties to the lowest, hist_tree_grower.cu:59-60), the record
// (WriteNode); at the last level also the weights of the node's leaves (k_tree_end's arithmetic) and the tree's
// record for the host.  grid L, 1024 threads, a wave per feature.
template <bool PAIR, bool F64>
__global__ void __launch_bounds__(1024)
k_ex_select(const Cand *__restrict__ best, const unsigned *__restrict__ node_first,
            const unsigned *__restrict__ node_items, unsigned max_items, int F,
            const unsigned char *__restrict__ active, const NodeSum *__restrict__ tot,
            const unsigned *__restrict__ seg_start, NodeSum *__restrict__ tot_next, unsigned *__restrict__ seg_next,
            SplitRec *__restrict__ split, int *__restrict__ t_fid, int *__restrict__ t_bin, float *__restrict__ t_gain,
            int L, int last, const int *__restrict__ shifts, GainParams gp, float eta, float *__restrict__ weights,
            const unsigned *__restrict__ overflow, uint32_t *__restrict__ record) {
  __shared__ Cand s_cand[16];
  __shared__ int s_fid[16];
  const int nd = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned first = node_first[nd];
  unsigned cnt = node_items[nd];
  if (cnt == 0xffffffffu) cnt = 0;
  Cand mine{};
  int fid = -1;
  for (int f = wave; f < F; f += 16) {
    if (active && !active[f]) continue;  // feature not sampled at this level
    const Cand *c = best + (size_t)f * max_items + first;
    // gains of candidates are positive: their bits order like the gains
    unsigned long long key = 0;
    unsigned at = 0;
    for (unsigned k = lane; k < cnt; k += 64) {
      const int bin = c[k].bin;
      if (bin < 0) continue;
      const unsigned long long x = ((unsigned long long)__float_as_uint(c[k].gain) << 32) | (unsigned)(bin + 1);
      if (x > key) {
        key = x;
        at = k;
      }
    }
    unsigned long long top = key;
    for (int o = 32; o > 0; o >>= 1) top = max(top, (unsigned long long)__shfl_xor(top, o));
    if (top == 0) continue;  // uniform
    if (fid >= 0 && !(__uint_as_float((unsigned)(top >> 32)) > mine.gain)) continue;
    // (the places of one node change to every rank once: one lane has the key)
    const int from = __ffsll((unsigned long long)__ballot(key == top)) - 1;
    mine = c[__builtin_amdgcn_readfirstlane(__shfl(at, from))];
    fid = f;
  }
  if (lane == 0) {
    s_cand[wave] = mine;
    s_fid[wave] = fid;
  }
  __syncthreads();
  const int internal = 2 * L - 1;
  if (last) {  // the nodes above the last level
    for (int i = nd * 1024 + (int)threadIdx.x; i < L - 1; i += L * 1024) {
      record[i] = (uint32_t)t_fid[i];
      record[internal + i] = (uint32_t)t_bin[i];
      record[2 * internal + i] = __float_as_uint(t_gain[i]);
    }
  }
  if (threadIdx.x != 0) return;
  for (int k = 1; k < 16; ++k) {
    if (s_fid[k] < 0) continue;
    if (fid < 0 || s_cand[k].gain > mine.gain || (s_cand[k].gain == mine.gain && s_fid[k] < fid)) {
      mine = s_cand[k];
      fid = s_fid[k];
    }
  }
  const NodeSum t = tot[nd];
  const SplitRec s = WriteNode(nd, t, mine.gain, fid, mine.bin, mine.left.g, mine.left.h, mine.left.c, seg_start, tot_next,
                               seg_next, split, t_fid, t_bin, t_gain, L - 1);
  if (!last) return;
  const int sg = shifts[0], sh = shifts[1];
  const double GL = FromFixed<F64>(s.left.g, sg), HL = PAIR ? FromFixed<F64>(s.left.h, sh) : 0.0;
  const double GP = FromFixed<F64>(t.g, sg), HP = PAIR ? FromFixed<F64>(t.h, sh) : 0.0;
  double GR, HR;
  if (F64) {
    GR = GP - GL;
    HR = HP - HL;
  } else {
    GR = (double)((float)GP - (float)GL);
    HR = (double)((float)HP - (float)HL);
  }
  const float wl = LeafWeight<PAIR, F64>(GL, HL, s.left.c, gp) * eta;
  const float wr = LeafWeight<PAIR, F64>(GR, HR, t.c - s.left.c, gp) * eta;
  const int at = L - 1 + nd;
  weights[2 * nd] = wl;
  weights[2 * nd + 1] = wr;
  record[at] = (uint32_t)(s.fid < 0 ? 0 : s.fid);
  record[internal + at] = (uint32_t)(s.fid < 0 ? -1 : s.bin);
  record[2 * internal + at] = __float_as_uint(s.gain);
  record[3 * internal + 2 * nd] = __float_as_uint(wl);
  record[3 * internal + 2 * nd + 1] = __float_as_uint(wr);
  if (nd == 0) record[3 * internal + 2 * L] = *overflow;
}

__device__ __forceinline__ bool ExGoesRight(const unsigned *__restrict__ ranks, size_t stride,
                                            const SplitRec *__restrict__ split, unsigned nd, size_t i) {
  const SplitRec s = split[nd];
  return s.fid >= 0 && ranks[(size_t)s.fid * stride + i] > (unsigned)s.bin;
}

// Every row to its child: node_of[row] = 2 * node + (rank of the split feature > split rank).
// went_right: one bit per row (64 rows per word), small enough to stay in L2 while the lists are
// partitioned.  ranks: [F][stride] by row.  The first block of the grid plans the children's level (`next`) instead, the
// others also clear its sums.
__global__ void __launch_bounds__(1024)
k_ex_decide(const unsigned *__restrict__ ranks, size_t stride, const SplitRec *__restrict__ split,
            unsigned *__restrict__ node_of, unsigned long long *__restrict__ went_right, size_t n, int root,
            const NodeSum *__restrict__ tot_next, const unsigned *__restrict__ seg_next, int L, const ExPlan next,
            unsigned grid_items, unsigned max_items, int F, unsigned *__restrict__ overflow) {
  if (blockIdx.x == 0) {
    PlanBody(tot_next, seg_next, 2 * L, 0, kExItem, next.work, next.n_work, next.node_first, next.node_items, nullptr,
             grid_items, overflow);
    return;
  }
  const size_t at = (size_t)(blockIdx.x - 1) * 1024 + threadIdx.x, step = (size_t)(gridDim.x - 1) * 1024;
  for (size_t k = at; k < (size_t)F * max_items; k += step) next.part[k] = ExSum{0, 0};
  const size_t padded = (n + 63) / 64 * 64;
  for (size_t i = at; i < padded; i += step) {
    bool right = false;
    if (i < n) {
      const unsigned nd = root ? 0u : node_of[i];
      right = ExGoesRight(ranks, stride, split, nd, i);
      node_of[i] = 2 * nd + (right ? 1u : 0u);
    }
    const unsigned long long m = __ballot(right);
    if ((threadIdx.x & 63) == 0) went_right[i >> 6] = m;
  }
}

__device__ __forceinline__ unsigned ExGoesLeft(const unsigned long long *__restrict__ went_right, unsigned id) {
  return (unsigned)(~(went_right[id >> 6] >> (id & 63u)) & 1ull);
}

// grid (items, F): rows of every piece that go left; left_bits: for every thread of every piece
// the decisions of its kExPer places (bit j: place j goes left), which the partition reads back
// instead of looking the rows up again.
__global__ void __launch_bounds__(kExThreads)
k_ex_count(const unsigned *__restrict__ ids, size_t stride, const unsigned long long *__restrict__ went_right,
           const ExPlan plan, unsigned *__restrict__ lefts,
           uint8_t *__restrict__ left_bits, unsigned max_items) {
  static_assert(kExPer == 8, "one byte of decisions per thread");
  __shared__ unsigned s_wave[kExThreads / 64];
  const unsigned w = blockIdx.x, f = blockIdx.y;
  if (w >= *plan.n_work) return;
  const WorkItem it = plan.work[w];
  const unsigned p0 = it.begin + threadIdx.x * kExPer;
  unsigned id[kExPer];
  ExLoad8(ids + (size_t)f * stride, p0, it.end, 0u, id);
  unsigned bits = 0;
#pragma unroll
  for (int j = 0; j < kExPer; ++j)
    if (p0 + j < it.end) bits |= ExGoesLeft(went_right, id[j]) << j;
  left_bits[((size_t)f * max_items + w) * kExThreads + threadIdx.x] = (uint8_t)bits;
  unsigned total;
  ExBlockScan((unsigned)__builtin_popcount(bits), s_wave, &total);
  if (threadIdx.x == 0) lefts[(size_t)f * max_items + w] = total;
}

// grid (items, F): the stable partition of every piece into the lists of the two children, with
// the rank and the gradients of every row next to its id (without hessians or with packed gradients the lists hold
// one word of gradients, else h beside g).  The piece is put in order in LDS
// (the rows that go left, then the others) and written out from there, so that the stores of a
// wave are consecutive; the sums of the gradients over the pieces of the children's lists (`next`) are made on the way: either part
// of the piece lies in two of them at most, and a wave writes 512 neighbouring places.  (A pass of its own over the new
// lists took 10 us a level at 400,000 rows x 20.)
// left_off: rows of the node's earlier pieces that go left, null: added up here from `lefts`;
// seg_start / seg_next: first place of the parents / of the children.
template <bool PAIR, bool PACK>
__global__ void __launch_bounds__(kExThreads)
k_ex_scatter(const ExLists ls, unsigned *__restrict__ ids_out, unsigned *__restrict__ ranks_out,
             float *__restrict__ g_out, float *__restrict__ h_out, size_t stride,
             const uint8_t *__restrict__ left_bits, const ExPlan plan, const unsigned *__restrict__ lefts,
             const unsigned *__restrict__ left_off, const unsigned *__restrict__ seg_start,
             const unsigned *__restrict__ seg_next, const int *__restrict__ shifts, const ExPlan next, unsigned max_items) {
  constexpr bool HARR = PAIR && !PACK;
  __shared__ unsigned s_wave[kExThreads / 64];
  __shared__ unsigned s_id[kExItem], s_rk[kExItem];
  __shared__ float s_g[kExItem], s_h[HARR ? kExItem : 1];
  const unsigned w = blockIdx.x, f = blockIdx.y;
  if (w >= *plan.n_work) return;
  const WorkItem it = plan.work[w];
  const size_t fbase = (size_t)f * stride;
  const unsigned p0 = it.begin + threadIdx.x * kExPer;
  unsigned id[kExPer], rk[kExPer];
  float gv[kExPer], hv[kExPer];
  ExLoad8(ls.ids + fbase, p0, it.end, 0u, id);
  ExLoad8(ls.ranks + fbase, p0, it.end, 0u, rk);
  ExLoad8(ls.g + fbase, p0, it.end, 0.0f, gv);
  if (HARR) ExLoad8(ls.h + fbase, p0, it.end, 0.0f, hv);
  const unsigned bits = left_bits[((size_t)f * max_items + w) * kExThreads + threadIdx.x];
  unsigned before = 0;
  if (left_off != nullptr) {  // uniform
    before = left_off[(size_t)f * max_items + w];
  } else {
    for (unsigned k = it.first + (threadIdx.x & 63); k < w; k += 64) before += lefts[(size_t)f * max_items + k];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
  }
  const unsigned mine = (unsigned)__builtin_popcount(bits);
  unsigned total;
  const unsigned incl = ExBlockScan(mine, s_wave, &total);
  // places of this thread's rows in the ordered piece
  unsigned l_at = incl - mine;
  unsigned r_at = total + threadIdx.x * kExPer - l_at;
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    if (p0 + j < it.end) {
      const unsigned at = ((bits >> j) & 1u) ? l_at++ : r_at++;
      s_id[at] = id[j];
      s_rk[at] = rk[j];
      s_g[at] = gv[j];
      if (HARR) s_h[at] = hv[j];
    }
  }
  __syncthreads();
  const unsigned count = it.end - it.begin;
  // first place of either part, and how many of its rows lie in the first of its work items (cut as PlanBody cuts
  // them: from the child's start rounded down to 64)
  unsigned to[2], in_first[2], item[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const unsigned child = 2 * it.node + c, start = seg_next[child], origin = start & ~63u;
    to[c] = c == 0 ? start + before : start + (it.begin - seg_start[it.node]) - before;
    const unsigned k = (to[c] - origin) / kExItem;
    in_first[c] = origin + (k + 1) * kExItem - to[c];
    item[c] = next.node_first[child] + k;
  }
  const int sg = shifts[0], sh = shifts[1], lane = threadIdx.x & 63;
  long long g_sum[4] = {0, 0, 0, 0}, h_sum[4] = {0, 0, 0, 0};
  unsigned seen = 0;
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    const unsigned k = (threadIdx.x >> 6) * (64 * kExPer) + j * 64 + lane;
    if (k < count) {
      const bool right = k >= total;
      const unsigned i = right ? k - total : k;
      const size_t at = fbase + (right ? to[1] : to[0]) + i;
      const float g0 = s_g[k], h0 = HARR ? s_h[k] : 0.0f;
      ids_out[at] = s_id[k];
      ranks_out[at] = s_rk[k];
      g_out[at] = g0;
      if (HARR) h_out[at] = h0;
      float g1 = g0, h1 = h0;
      if (PACK) UnpackGrad(g0, &g1, &h1);
      const long long gq = ToFixed(g1, sg), hq = PAIR ? ToFixed(h1, sh) : 0;
      const unsigned slot = (right ? 2u : 0u) + (i >= (right ? in_first[1] : in_first[0]) ? 1u : 0u);
      seen |= 1u << slot;
#pragma unroll
      for (unsigned q = 0; q < 4; ++q) {
        g_sum[q] += slot == q ? gq : 0;
        if (PAIR) h_sum[q] += slot == q ? hq : 0;
      }
    }
  }
#pragma unroll
  for (unsigned q = 0; q < 4; ++q) {
    if (__ballot((seen >> q) & 1u) == 0ull) continue;  // uniform
    const long long gs = WaveSumLL(g_sum[q]), hs = PAIR ? WaveSumLL(h_sum[q]) : 0;
    if (lane == 0) {
      ExSum *p = &next.part[(size_t)f * max_items + item[q >> 1] + (q & 1u)];
      atomicAdd(reinterpret_cast<unsigned long long *>(&p->g), (unsigned long long)gs);
      if (PAIR) atomicAdd(reinterpret_cast<unsigned long long *>(&p->h), (unsigned long long)hs);
    }
  }
}

// (g, h) of every row side by side, so that one access fetches both.
__global__ void k_ex_pair(const float *__restrict__ g, const float *__restrict__ h, float2 *__restrict__ gh, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    gh[i] = make_float2(g[i], h[i]);
}

// grid (ceil(n / kExItem), F): the gradients of this tree in the order of the root's lists, and their sums over the root's
// work items, which are the blocks of this grid.
template <bool PAIR, bool PACK>
__global__ void __launch_bounds__(kExThreads)
k_ex_gather(const unsigned *__restrict__ ids, size_t stride, const float *__restrict__ g,
            const float2 *__restrict__ gh, float *__restrict__ g_out, float *__restrict__ h_out, size_t n,
            const int *__restrict__ shifts, ExSum *__restrict__ part, unsigned max_items) {
  __shared__ long long s_sums[kExThreads / 64][2];
  const size_t fbase = (size_t)blockIdx.y * stride;
  const int sg = shifts[0], sh = shifts[1];
  long long sum[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < kExPer; ++j) {
    const size_t p = (size_t)blockIdx.x * kExItem + (size_t)j * kExThreads + threadIdx.x;
    if (p < n) {
      const unsigned id = ids[fbase + p];
      float g1, h1 = 0.0f;
      if (PAIR && !PACK) {
        const float2 v = gh[id];
        g1 = v.x;
        h1 = v.y;
        g_out[fbase + p] = g1;
        h_out[fbase + p] = h1;
      } else {
        g1 = g[id];
        g_out[fbase + p] = g1;
        if (PACK) UnpackGrad(g1, &g1, &h1);
      }
      sum[0] += ToFixed(g1, sg);
      if (PAIR) sum[1] += ToFixed(h1, sh);
    }
  }
  ExBlockSums(sum, s_sums);
  if (threadIdx.x == 0) part[(size_t)blockIdx.y * max_items + blockIdx.x] = ExSum{sum[0], sum[1]};
}

// End of a tree: every row to its leaf, the leaf's weight to its prediction (update_by_last_tree,
// src/core/garden.cu:45-76) and, when NEXT_GRAD is not 0, the gradients of the next round, as k_final writes them
// (1 = squared, with the largest |g| of every workgroup; 2 = logistic, packed when h is null).
template <int NEXT_GRAD>
__global__ void __launch_bounds__(256)
k_ex_final(const unsigned *__restrict__ ranks, size_t stride, const SplitRec *__restrict__ split,
           const unsigned *__restrict__ node_of, int root, const float *__restrict__ weights, float *__restrict__ yhat,
           unsigned *__restrict__ leaf_of, size_t n, const float *__restrict__ y, float *__restrict__ g,
           float *__restrict__ h, float *__restrict__ gmax_parts) {
  float m = 0.0f;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const unsigned nd = root ? 0u : node_of[i];
    const unsigned leaf = 2 * nd + (ExGoesRight(ranks, stride, split, nd, i) ? 1u : 0u);
    leaf_of[i] = leaf;
    const float yh = yhat[i] + weights[leaf];
    yhat[i] = yh;
    if (NEXT_GRAD == 1) {
      const float v = y[i] - yh;
      g[i] = v;
      const float a = fabsf(v);
      if (a > m) m = a;
    } else if (NEXT_GRAD == 2) {
      const float s = SigmoidF(yh), yv = y[i];
      if (h != nullptr) {
        g[i] = yv - s;
        h[i] = s * (1.0f - s);
      } else {
        g[i] = PackGrad(s, yv);
      }
    }
  }
  if (NEXT_GRAD == 1) {
    m = BlockMaxF(m);
    if (threadIdx.x == 0) gmax_parts[blockIdx.x] = m;
  }
}

}  // namespace
}  // namespace arb
#endif  // ARBORETUM_AMD_KERNELS_EXACT_H_
