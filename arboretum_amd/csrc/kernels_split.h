// Split search: prefix scan and gain per feature, best feature per node.
#ifndef ARBORETUM_AMD_KERNELS_SPLIT_H_
#define ARBORETUM_AMD_KERNELS_SPLIT_H_
#include "device_common.h"
#include "kernels_plan.h"

namespace arb {

// The best candidate of one feature of a node (bin -1: none).
struct Cand {
  float gain;
  int bin;
  NodeSum left;
};

// What a fused pass over the rows of a level's nodes needs to select the splits of those nodes
// itself, in its prologue, from the per-feature candidates of the split scan (k_split_scan)
// instead of reading them from a selection kernel launched before it: one launch less per level
// on the critical path.  Every workgroup of the pass selects for ITS node; the node's first work
// item also writes the node's record.  cand == null: the splits are read from `split` as before.
struct LevelScan {
  const Cand *cand;
  int F, L;
  NodeSum *tot_next;
  unsigned *seg_next;
  SplitRec *split;
  int *t_fid, *t_bin;
  float *t_gain;
  int heap_off;
  const unsigned char *active;
  const unsigned *node_first;         // first work item of every node: that item writes the node's record
  unsigned long long *rows_scanned;   // advanced by the rows of the smaller side of every split
};

namespace {

// --------------------------------------------------------------- split scan

// The candidates among 64 BPL neighbouring bins of a feature from `chunk` on, BPL of them in every lane (sums per bin; overwritten).
// carry: the sums below them, and then with them.
template <bool PAIR, bool F64, int BPL>
__device__ __forceinline__ void ScanChunk(long long (&g4)[BPL], long long (&h4)[BPL], unsigned long long (&c4)[BPL],
                                          int chunk, int lane, double GT, double HT, const NodeSum &t, int sg, int sh,
                                          const GainParams &gp, int hist_size, NodeSum *carry, Cand *best) {
#pragma unroll
  for (int j = 1; j < BPL; ++j) {
    g4[j] += g4[j - 1];
    h4[j] += h4[j - 1];
    c4[j] += c4[j - 1];
  }
  long long ig = g4[BPL - 1], ih = h4[BPL - 1];
  unsigned long long ic = c4[BPL - 1];
  for (int off = 1; off < 64; off <<= 1) {
    const long long og = __shfl_up(ig, off);
    const long long oh = PAIR ? __shfl_up(ih, off) : 0;
    const unsigned long long oc = __shfl_up(ic, off);
    if (lane >= off) {
      ig += og;
      ih += oh;
      ic += oc;
    }
  }
  const long long eg = carry->g + ig - g4[BPL - 1], eh = carry->h + ih - h4[BPL - 1];
  const unsigned long long ec = carry->c + ic - c4[BPL - 1];
#pragma unroll
  for (int j = 0; j < BPL; ++j) {
    const int bin = chunk + lane * BPL + j;
    if (bin < hist_size) {
      const long long lg = eg + g4[j], lh = eh + h4[j];
      const unsigned long long lc = ec + c4[j];
      const double GL = FromFixed<F64>(lg, sg);
      const double HL = PAIR ? FromFixed<F64>(lh, sh) : 0.0;
      const float gn = SplitGain<PAIR, F64>(GL, HL, lc, GT, HT, t.c, gp);
      if (gn > 0.0f && gn >= best->gain) {
        best->gain = gn;
        best->bin = bin;
        best->left.g = lg;
        best->left.h = lh;
        best->left.c = lc;
      }
    }
  }
  carry->g += __shfl(ig, 63);
  if (PAIR) carry->h += __shfl(ih, 63);
  carry->c += __shfl(ic, 63);
}
// The best candidate of a wave in every lane: highest gain, ties to the highest bin (bins differ).
template <bool PAIR>
__device__ __forceinline__ void BestOfWave(Cand *best) {
  // one key, then the winner's sums
  unsigned long long key = best->bin < 0 ? 0ull : ((unsigned long long)__float_as_uint(best->gain) << 32) | (unsigned)(best->bin + 1);
  unsigned long long top = key;
  for (int off = 32; off > 0; off >>= 1) top = max(top, (unsigned long long)__shfl_xor(top, off));
  if (top != 0) {  // uniform
    const int from = __ffsll((unsigned long long)__ballot(key == top)) - 1;  // (keys differ by their bins)
    best->gain = __shfl(best->gain, from);
    best->bin = __shfl(best->bin, from);
    best->left.g = __shfl(best->left.g, from);
    best->left.h = PAIR ? __shfl(best->left.h, from) : 0;
    best->left.c = __shfl(best->left.c, from);
  }
}

// One wave scans one (feature, node): inclusive prefix over the slots, gain
// per bin < hist_size, arg-max with ties to the HIGHEST bin (builder.h:39-49),
// only gains > 0 (hist_tree_grower.cu:31).  `first` is the index of the
// feature's slot 0 in the histogram arrays.  The result is valid in lane 0.
// BPL: neighbouring bins per lane, 64 BPL bins at a time.  The gains of a lane's
// bins are double-precision arithmetic one after the other, so a feature of 64
// bins is scanned with one bin per lane (with four, 16 lanes did the work of 64).
template <bool PAIR, bool F64, int BPL>
__device__ __forceinline__ Cand ScanFeature(const long long *__restrict__ hg, const long long *__restrict__ hh,
                                            const unsigned long long *__restrict__ hc, size_t first, int slots,
                                            const NodeSum &t, const int *__restrict__ shifts,
                                            const GainParams &gp, int hist_size, int lane) {
  Cand best;
  best.gain = 0.0f;
  best.bin = -1;
  best.left.g = best.left.h = 0;
  best.left.c = 0;
  if (t.c != 0) {
    const int sg = shifts[0], sh = shifts[1];
    const double GT = FromFixed<F64>(t.g, sg);
    const double HT = PAIR ? FromFixed<F64>(t.h, sh) : 0.0;
    NodeSum carry{0, 0, 0};  // sums of the slots below the current chunk
    for (int chunk = 0; chunk < slots && chunk < hist_size; chunk += 64 * BPL) {
      const size_t base = first + chunk + lane * BPL;
      long long g4[BPL], h4[BPL];
      unsigned long long c4[BPL];
#pragma unroll
      for (int j = 0; j < BPL; ++j) g4[j] = h4[j] = 0, c4[j] = 0;
      // lanes whose slots all lie at or past hist_size (missing values, unused slots) hold no
      // candidate and are in no candidate's prefix: they read nothing
      if (chunk + lane * BPL < hist_size) {
#pragma unroll
        for (int j = 0; j < BPL; ++j) {
          g4[j] = hg[base + j];
          h4[j] = PAIR ? hh[base + j] : 0;
          c4[j] = hc[base + j];
        }
      }
      ScanChunk<PAIR, F64, BPL>(g4, h4, c4, chunk, lane, GT, HT, t, sg, sh, gp, hist_size, &carry, &best);
    }
    BestOfWave<PAIR>(&best);
  }
  return best;
}

// grid (ceil(F / 4), L), 256 threads: one wave per (feature, node), candidates to `cand`.
// root_sum (the root level): the gradient totals of the root are the sum over the slots of feature 0
// of its histogram (every row, NaN included, sits in exactly one slot; replaces the reduction over the
// gradient array of garden.cu:432-435).  Every wave makes that sum for itself, a kilobyte or two out of
// the cache, and one writes it to tot[0]: no kernel of its own in between.  hi_cell > 0: the cell of
// feature 0's bin 256 (matrices with a ninth-bit word).
template <bool PAIR, bool F64, int BPL>
__global__ void __launch_bounds__(256)
k_split_scan(const long long *__restrict__ hg, const long long *__restrict__ hh,
             const unsigned long long *__restrict__ hc, int nbin_total, int F, int slots,
             NodeSum *__restrict__ tot, const int *__restrict__ shifts, GainParams gp,
             int hist_size, Cand *__restrict__ cand, int root_sum, int hi_cell) {
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6), nd = blockIdx.y, lane = threadIdx.x & 63;
  if (f >= F) return;
  NodeSum t = tot[nd];
  if (root_sum) {
    long long a = 0, b = 0;
    for (int i = lane; i < slots; i += 64) {
      a += hg[i];
      if (PAIR) b += hh[i];
    }
    if (hi_cell > 0 && lane == 0) {
      a += hg[hi_cell];
      if (PAIR) b += hh[hi_cell];
    }
    for (int off = 32; off > 0; off >>= 1) {
      a += __shfl_xor(a, off);
      if (PAIR) b += __shfl_xor(b, off);
    }
    t.g = a;
    t.h = b;
    if (f == 0 && lane == 0) {
      tot[0].g = a;
      tot[0].h = b;
    }
  }
  const Cand best = ScanFeature<PAIR, F64, BPL>(hg, hh, hc, (size_t)nd * nbin_total + (size_t)f * slots, slots, t, shifts,
                                                gp, hist_size, lane);
  if (lane == 0) cand[(size_t)nd * F + f] = best;
}

// The same for features of more than 256 bins (16-bit ids): a workgroup per feature and node, its four waves scan 256 bins
// each at a time.  (One wave, four times 256 bins one after the other: 13.9 us for 1000 bins x 20 features; 7.3.)
// grid (F, L), 256 threads.
template <bool PAIR, bool F64>
__global__ void __launch_bounds__(256)
k_split_scan_wide(const long long *__restrict__ hg, const long long *__restrict__ hh,
                  const unsigned long long *__restrict__ hc, int nbin_total, int F, int slots,
                  NodeSum *__restrict__ tot, const int *__restrict__ shifts, GainParams gp,
                  int hist_size, Cand *__restrict__ cand, int root_sum) {
  constexpr int BPL = 4, kWaves = 4;
  __shared__ NodeSum s_sum[kWaves];
  __shared__ Cand s_best[kWaves];
  const int f = blockIdx.x, nd = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  NodeSum t = tot[nd];
  if (root_sum) {
    long long a = 0, b = 0;
    for (int i = threadIdx.x; i < slots; i += 256) {
      a += hg[i];
      if (PAIR) b += hh[i];
    }
    a = WaveSumLL(a);
    b = PAIR ? WaveSumLL(b) : 0;
    if (lane == 0) s_sum[wave] = NodeSum{a, b, 0};
    __syncthreads();
    t.g = t.h = 0;
    for (int k = 0; k < kWaves; ++k) {
      t.g += s_sum[k].g;
      t.h += s_sum[k].h;
    }
    __syncthreads();
    if (f == 0 && threadIdx.x == 0) {
      tot[0].g = t.g;
      tot[0].h = t.h;
    }
  }
  const size_t first = (size_t)nd * nbin_total + (size_t)f * slots;
  const int sg = shifts[0], sh = shifts[1];
  const double GT = FromFixed<F64>(t.g, sg);
  const double HT = PAIR ? FromFixed<F64>(t.h, sh) : 0.0;
  Cand best;
  best.gain = 0.0f;
  best.bin = -1;
  best.left = NodeSum{0, 0, 0};
  NodeSum carry{0, 0, 0};  // of the slots below the current 1024
  for (int chunk = 0; chunk < slots && chunk < hist_size && t.c != 0; chunk += 64 * BPL * kWaves) {
    const int at = chunk + wave * 64 * BPL + lane * BPL;
    long long g4[BPL], h4[BPL];
    unsigned long long c4[BPL];
#pragma unroll
    for (int j = 0; j < BPL; ++j) {
      const bool on = at < hist_size;  // (slots is a multiple of BPL beyond hist_size)
      g4[j] = on ? hg[first + at + j] : 0;
      h4[j] = PAIR && on ? hh[first + at + j] : 0;
      c4[j] = on ? hc[first + at + j] : 0;
    }
#pragma unroll
    for (int j = 1; j < BPL; ++j) {
      g4[j] += g4[j - 1];
      h4[j] += h4[j - 1];
      c4[j] += c4[j - 1];
    }
    long long ig = g4[BPL - 1], ih = h4[BPL - 1];
    unsigned long long ic = c4[BPL - 1];
    for (int off = 1; off < 64; off <<= 1) {
      const long long og = __shfl_up(ig, off);
      const long long oh = PAIR ? __shfl_up(ih, off) : 0;
      const unsigned long long oc = __shfl_up(ic, off);
      if (lane >= off) {
        ig += og;
        ih += oh;
        ic += oc;
      }
    }
    __syncthreads();  // s_sum may still be read from the chunk before
    if (lane == 63) s_sum[wave] = NodeSum{ig, ih, ic};
    __syncthreads();
    NodeSum before = carry;
    for (int k = 0; k < kWaves; ++k) {
      const NodeSum x = s_sum[k];
      if (k < wave) {
        before.g += x.g;
        before.h += x.h;
        before.c += x.c;
      }
      carry.g += x.g;
      carry.h += x.h;
      carry.c += x.c;
    }
    const long long eg = before.g + ig - g4[BPL - 1], eh = before.h + ih - h4[BPL - 1];
    const unsigned long long ec = before.c + ic - c4[BPL - 1];
#pragma unroll
    for (int j = 0; j < BPL; ++j) {
      const int bin = at + j;
      if (bin < hist_size) {
        const long long lg = eg + g4[j], lh = eh + h4[j];
        const unsigned long long lc = ec + c4[j];
        const double GL = FromFixed<F64>(lg, sg);
        const double HL = PAIR ? FromFixed<F64>(lh, sh) : 0.0;
        const float gn = SplitGain<PAIR, F64>(GL, HL, lc, GT, HT, t.c, gp);
        if (gn > 0.0f && gn >= best.gain) {
          best.gain = gn;
          best.bin = bin;
          best.left = NodeSum{lg, lh, lc};
        }
      }
    }
  }
  // highest gain, ties to the highest bin
  const unsigned long long key = best.bin < 0 ? 0ull : ((unsigned long long)__float_as_uint(best.gain) << 32) | (unsigned)(best.bin + 1);
  unsigned long long top = key;
  for (int off = 32; off > 0; off >>= 1) top = max(top, (unsigned long long)__shfl_xor(top, off));
  if (lane == __ffsll((unsigned long long)__ballot(key == top)) - 1) s_best[wave] = best;
  __syncthreads();
  if (threadIdx.x != 0) return;
  best = s_best[0];
  for (int k = 1; k < kWaves; ++k)
    if (s_best[k].bin >= 0 && (best.bin < 0 || s_best[k].gain > best.gain ||
                               (s_best[k].gain == best.gain && s_best[k].bin > best.bin)))
      best = s_best[k];
  cand[(size_t)nd * F + f] = best;
}

// Record of one node from its best candidate (fid < 0: none, every row stays
// left): split, totals and row ranges of the two children, tree arrays.
__device__ __forceinline__ SplitRec WriteNode(int nd, const NodeSum &t, float gain, int fid, int bin, long long lg,
                                          long long lh, unsigned long long lc,
                                          const unsigned *__restrict__ seg_start, NodeSum *__restrict__ tot_next,
                                          unsigned *__restrict__ seg_next, SplitRec *__restrict__ split,
                                          int *__restrict__ t_fid, int *__restrict__ t_bin,
                                          float *__restrict__ t_gain, int heap_off) {
  SplitRec rec;
  rec.gain = fid < 0 ? 0.0f : gain;
  rec.fid = fid;
  rec.bin = fid < 0 ? -1 : bin;
  rec.pad = 0;
  rec.left = t;
  if (fid >= 0) {
    rec.left.g = lg;
    rec.left.h = lh;
    rec.left.c = lc;
  }
  split[nd] = rec;
  NodeSum r;
  r.g = t.g - rec.left.g;
  r.h = t.h - rec.left.h;
  r.c = t.c - rec.left.c;
  tot_next[2 * nd] = rec.left;
  tot_next[2 * nd + 1] = r;
  const unsigned start = seg_start[nd];
  seg_next[2 * nd] = start;
  seg_next[2 * nd + 1] = start + (unsigned)rec.left.c;
  t_fid[heap_off + nd] = rec.fid < 0 ? 0 : rec.fid;  // garden.cu:471-481
  t_bin[heap_off + nd] = rec.fid < 0 ? -1 : rec.bin;
  t_gain[heap_off + nd] = rec.gain;
  return rec;
}


// The best of a node's per-feature candidates over the features active at its level: the highest
// gain, ties to the lowest feature id (hist_tree_grower.cu:59-60).  One wave; every lane gets the
// feature (-1: no candidate) and the candidate.  Gains of candidates are positive, so their bits order
// like the gains, and one 64-bit maximum of (gain, ~feature) decides: two shuffles per step instead of
// one for every word of a candidate (2.4 -> 1.6 us of the prologue of a pass).
__device__ __forceinline__ int BestOfNode(const Cand *__restrict__ cand, int F, const unsigned char *__restrict__ active,
                                          int lane, Cand *best) {
  unsigned long long key = 0;  // larger than that of no candidate: the gain of a candidate is positive
  for (int f = lane; f < F; f += 64) {
    if (active && !active[f]) continue;  // feature not sampled at this level
    if (cand[f].bin < 0) continue;
    const unsigned long long k = ((unsigned long long)__float_as_uint(cand[f].gain) << 32) | (0xffffffffu - (unsigned)f);
    key = max(key, k);
  }
  for (int off = 32; off > 0; off >>= 1) key = max(key, (unsigned long long)__shfl_xor(key, off));
  best->gain = 0.0f;
  best->bin = -1;
  best->left.g = best->left.h = 0;
  best->left.c = 0;
  if (key == 0) return -1;  // uniform
  const int fid = (int)__builtin_amdgcn_readfirstlane(0xffffffffu - (unsigned)key);
  *best = cand[fid];
  return fid;
}

// Split of node nd (totals t) from its candidates: wave 0 of the workgroup keeps the candidate
// with the highest gain, ties to the lowest feature id (hist_tree_grower.cu:59-60), over the
// features active at this level; every thread returns the node's record.  `write`: this
// workgroup also stores the record, the children's totals and row ranges and the tree arrays
// (WriteNode).  Called by all threads of the workgroup; s_rec holds one record.
__device__ __forceinline__ SplitRec SelectInPass(const LevelScan &a, int nd, const NodeSum &t,
                                                 const unsigned *__restrict__ seg_start, bool write,
                                                 SplitRec *s_rec) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave == 0) {
    Cand c;
    c.gain = 0.0f;
    c.bin = -1;
    c.left = NodeSum{0, 0, 0};
    const int fid = t.c == 0 ? -1 : BestOfNode(a.cand + (size_t)nd * a.F, a.F, a.active, lane, &c);
    const float gain = c.gain;
    const int bin = c.bin;
    const long long lg = c.left.g, lh = c.left.h;
    const unsigned long long lc = c.left.c;
    if (lane == 0) {
      SplitRec rec;
      if (write) {
        rec = WriteNode(nd, t, gain, fid, bin, lg, lh, lc, seg_start, a.tot_next, a.seg_next, a.split, a.t_fid,
                        a.t_bin, a.t_gain, a.heap_off);
        if (a.rows_scanned && t.c != 0) {
          const unsigned long long cl = fid < 0 ? t.c : lc;
          atomicAdd(a.rows_scanned, min(cl, t.c - cl));
        }
      } else {
        rec.gain = fid < 0 ? 0.0f : gain;
        rec.fid = fid;
        rec.bin = fid < 0 ? -1 : bin;
        rec.pad = 0;
        rec.left = t;
        if (fid >= 0) {
          rec.left.g = lg;
          rec.left.h = lh;
          rec.left.c = lc;
        }
      }
      *s_rec = rec;
    }
  }
  __syncthreads();
  // the record as wave-uniform values (it steers the whole pass)
  SplitRec r;
  r.gain = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(s_rec->gain)));
  r.fid = __builtin_amdgcn_readfirstlane(s_rec->fid);
  r.bin = __builtin_amdgcn_readfirstlane(s_rec->bin);
  r.pad = 0;
  const unsigned long long *p = reinterpret_cast<const unsigned long long *>(&s_rec->left);
  unsigned long long v[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)p[k]);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(p[k] >> 32));
    v[k] = ((unsigned long long)hi << 32) | lo;
  }
  r.left.g = (long long)v[0];
  r.left.h = (long long)v[1];
  r.left.c = v[2];
  return r;
}

// Records of the nodes of a level that hold no row (no work item of the pass stands for them):
// not split, both children empty.  Called by one workgroup.
__device__ __forceinline__ void WriteEmptyNodes(const LevelScan &a, const NodeSum *__restrict__ tot,
                                                const unsigned *__restrict__ seg_start) {
  for (int nd = threadIdx.x; nd < a.L; nd += blockDim.x) {
    const NodeSum t = tot[nd];
    if (t.c == 0)
      WriteNode(nd, t, 0.0f, -1, -1, 0, 0, 0, seg_start, a.tot_next, a.seg_next, a.split, a.t_fid, a.t_bin, a.t_gain,
                a.heap_off);
  }
}


// One thread per node: best candidate over the features active at this level
// (higher gain, then lower feature id: hist_tree_grower.cu:59-60), children
// totals and row ranges, node record.  A node without a candidate keeps every
// row left.
// One wave per node: lane l looks at features l, l + 64, ...; the wave keeps
// the candidate with the highest gain, ties to the lowest feature id.
__device__ __forceinline__ SplitRec SelectNode(int nd, int lane, const Cand *__restrict__ cand, int F,
                                           const NodeSum *__restrict__ tot,
                                           const unsigned *__restrict__ seg_start,
                                           NodeSum *tot_next, unsigned *seg_next,
                                           SplitRec *__restrict__ split, int *__restrict__ t_fid,
                                           int *__restrict__ t_bin, float *__restrict__ t_gain, int heap_off,
                                           const unsigned char *__restrict__ active) {
  const NodeSum t = tot[nd];
  Cand c;
  c.gain = 0.0f;
  c.bin = -1;
  c.left = NodeSum{0, 0, 0};
  const int fid = t.c == 0 ? -1 : BestOfNode(cand + (size_t)nd * F, F, active, lane, &c);
  SplitRec rec{};
  if (lane == 0)
    rec = WriteNode(nd, t, c.gain, fid, c.bin, c.left.g, c.left.h, c.left.c, seg_start, tot_next, seg_next, split, t_fid,
                    t_bin, t_gain, heap_off);
  return rec;  // valid in lane 0
}

// grid ceil(L / 16), 1024 threads: one wave per node.  rows_scanned (optional): advanced by the rows of
// the smaller side of every split.
__global__ void __launch_bounds__(1024)
k_split_select(const Cand *__restrict__ cand, int F, int L, const NodeSum *__restrict__ tot,
               const unsigned *__restrict__ seg_start, NodeSum *__restrict__ tot_next,
               unsigned *__restrict__ seg_next, SplitRec *__restrict__ split, int *__restrict__ t_fid,
               int *__restrict__ t_bin, float *__restrict__ t_gain, int heap_off,
               const unsigned char *__restrict__ active, unsigned long long *__restrict__ rows_scanned) {
  const int nd = blockIdx.x * 16 + (threadIdx.x >> 6);
  if (nd >= L) return;
  const SplitRec r = SelectNode(nd, threadIdx.x & 63, cand, F, tot, seg_start, tot_next, seg_next, split, t_fid, t_bin,
                                t_gain, heap_off, active);
  if (rows_scanned && (threadIdx.x & 63) == 0) {
    const unsigned long long c = tot[nd].c;
    if (c != 0) atomicAdd(rows_scanned, min(r.left.c, c - r.left.c));
  }
}

// Splits of a level's nodes and the work plan of the children's histograms, made by the partition that
// follows the split scan on the paths with stand-alone histogram launches: every workgroup selects for
// its own node (SplitOf), and one more block of the grid (the first one) selects for all of them, writes
// their records and plans (SelectAndPlan; `select`, balance_cus: PlanBody's).  A launch of its own
// stood between scan and partition for 6.5 us a level, and the partition takes 3 us longer for it while its work items fit
// two rounds of the chip.  One workgroup does it beside the partition while the level has few nodes.  cand == null: the splits
// have been selected by k_split_select (HipTreeBuilder::SelectInPartition); the kernels of large items have an instance for
// that (SELECT = false) without the planner's 16 KB of LDS and a third of the scalar registers: 50 M x 200, max_depth
// 10: 3.76 ms a tree, 4.11 by the other one.
struct SelectPlan {
  const Cand *cand = nullptr;
  int F = 0, L = 0;
  const NodeSum *tot = nullptr;
  const unsigned *seg_start = nullptr;
  NodeSum *tot_next = nullptr;
  unsigned *seg_next = nullptr;
  SplitRec *split = nullptr;
  int *t_fid = nullptr, *t_bin = nullptr;
  float *t_gain = nullptr;
  const unsigned char *active = nullptr;
  int select = 0;
  unsigned rows_per_item = 0;
  WorkItem *work = nullptr;
  unsigned *n_work = nullptr, *node_first = nullptr, *node_items = nullptr;
  unsigned long long *rows_scanned = nullptr;
  unsigned max_items = 0;
  unsigned *overflow = nullptr;
  unsigned balance_cus = 0;
};
constexpr int kSelectPlanNodes = 64;  // most nodes of a level whose partition selects and plans

__device__ __forceinline__ void SelectAndPlan(const SelectPlan &a) {
  for (int nd = threadIdx.x >> 6; nd < a.L; nd += blockDim.x / 64)
    SelectNode(nd, threadIdx.x & 63, a.cand, a.F, a.tot, a.seg_start, a.tot_next, a.seg_next, a.split, a.t_fid, a.t_bin,
               a.t_gain, a.L - 1, a.active);
  __syncthreads();  // the children's totals and ranges written above are read by the plan
  PlanBody(a.tot_next, a.seg_next, 2 * a.L, a.select, a.rows_per_item, a.work, a.n_work, a.node_first, a.node_items,
           a.rows_scanned, a.max_items, a.overflow, nullptr, a.balance_cus);
}
// Called by all threads of the workgroup.
__device__ __forceinline__ SplitRec SplitOf(const SelectPlan &a, int nd, const SplitRec *__restrict__ split) {
  if (a.cand == nullptr) return split[nd];  // uniform
  __shared__ SplitRec s_rec;
  LevelScan scan{};
  scan.cand = a.cand;
  scan.F = a.F;
  scan.active = a.active;
  return SelectInPass(scan, nd, a.tot[nd], a.seg_start, false, &s_rec);
}

}  // namespace
}  // namespace arb
#endif  // ARBORETUM_AMD_KERNELS_SPLIT_H_
