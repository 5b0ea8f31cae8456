// Batch prediction on the GPU: the tree walks of RegTree::Predict /
// Garden::Predict (src/core/garden.h:70-90, src/core/garden.cu:643-657) for a
// float matrix (or a pre-quantised one, whose bin ids are compared as floats
// like the host walk does).  The arithmetic is the host walk's: `x < threshold`
// goes left (NaN right), the leaf weights of one label are added in tree order
// in fp32, so the sums are bit-identical to the host path.  The link function
// stays with the caller.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <limits>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "booster.h"
#include "memory_pool.h"
#include "parallel.h"
#include "staging.h"

namespace arb {
namespace {

#define HIP_OK(expr)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + " in " #expr); \
  } while (0)

constexpr unsigned kWalkThreads = 1024;
constexpr size_t kWalkLds = 159 * 1024;           // of the 160 KB of a CU: one workgroup of 16 waves has it
constexpr size_t kTreeLds = 40 * 1024;            // trees staged at a time when rows are many
constexpr unsigned kAhead = 5;                    // words per thread fetched while the chunk before is walked
constexpr unsigned kChains = 4;                   // trees a thread walks side by side
constexpr size_t kBlockBytes = (size_t)32 << 20;  // device block of rows that are not kept on the device
constexpr size_t kMostModelBytes = (size_t)1 << 31;  // (trees are addressed by 32-bit byte offsets)

// A tree as 8-byte words: its 2^(depth-1) - 1 nodes (feature, threshold bits) in heap order, then its
// 2^(depth-1) leaf weights, two to a word.
struct TreeRef {
  unsigned off, depth, label, unused;
};

size_t TreeWords(const RegTree &t) { return t.fid.size() + t.weights.size() / 2; }

// Where a row's feature values come from.
enum Source {
  kFloatRows = 0,  // float rows [n][F]
  kByteRows = 1,   // pre-quantised rows [n][F] of uint8 bin ids
  kQuadCols = 2    // pre-quantised quad columns [Q][ld]: four uint8 bin ids per word
};

struct Walk {
  const void *base;
  size_t ld;               // kQuadCols
  unsigned n, F;           // rows at `base`, features
  unsigned rows_log;       // log2 of the rows of a workgroup, 6 ... 10
  const uint2 *words;
  const TreeRef *refs;     // n_trees of them in order of labels, and one more whose `off` is the end
  unsigned n_trees, per_chunk, labels;
  unsigned tree_words;     // != 0: every tree has so many words and the depth `depth`
  unsigned depth;
  unsigned words_at, leaf_at;  // bytes: where in the LDS the trees and the leaf weights found stand
  float init;
  float *out;              // [labels][out_ld], at the first of the n rows
  size_t out_ld;
};

// The LDS by byte address: a 32-bit register is the whole address of a read.
template <typename T>
__device__ __forceinline__ T LdsAt(unsigned at) {
  return *(const __attribute__((address_space(3))) T *)(uintptr_t)at;
}
__device__ __forceinline__ unsigned LdsAddress(const unsigned char *p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char *)p;
}

template <int SRC>
struct Values {
  typedef unsigned char T;
};
template <>
struct Values<kFloatRows> {
  typedef float T;
};

// Value of feature f of the thread's row: from the LDS tile [F][R], or from memory.
template <int SRC, bool TILE>
struct Fetch {
  unsigned R, r;  // bytes of R elements, LDS address of the row's value of feature 0
  const Walk &a;
  size_t row;
  __device__ __forceinline__ float operator()(unsigned f) const {
    if (TILE) return (float)LdsAt<typename Values<SRC>::T>(__umul24(f, R) + r);
    if (SRC == kQuadCols)
      return (float)((static_cast<const uint32_t *>(a.base)[(size_t)(f >> 2) * a.ld + row] >> (8u * (f & 3u))) & 255u);
    return (float)static_cast<const typename Values<SRC>::T *>(a.base)[row * a.F + f];
  }
};

// (no class type: it is read through a pointer of an address space)
typedef unsigned Node __attribute__((ext_vector_type(2)));

// N trees walked side by side: their chains of a node and a value read per level overlap.  w: where
// the trees start, LDS addresses or bytes from `words`.  The children of the node at byte p of its tree are at
// 2 p + 8 and 2 p + 16, so there at 2 at - w + 8 (16): four vector instructions a level
// beside the two reads (counting in nodes takes nine, and the walk is as much bound by them as by the LDS).
template <bool IN_LDS, int N, typename F>
__device__ __forceinline__ void WalkTrees(const unsigned char *words, const unsigned (&w)[N], unsigned depth,
                                          const F &fetch, float *leaf) {
  unsigned at[N], left[N], right[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    at[k] = w[k];
    left[k] = 8u - w[k];
    right[k] = 16u - w[k];
    asm("" : "+v"(left[k]), "+v"(right[k]));  // (registers, not 8 and 16 less w again on every level)
  }
  for (unsigned j = 1; j < depth; ++j) {
    Node nd[N];
    float v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) nd[k] = IN_LDS ? LdsAt<Node>(at[k]) : *reinterpret_cast<const Node *>(words + at[k]);
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = fetch(nd[k].x);
#pragma unroll
    for (int k = 0; k < N; ++k) at[k] = (at[k] << 1) + (v[k] < __uint_as_float(nd[k].y) ? left[k] : right[k]);
  }
  // node id = (at - w) / 8; its leaf id - nodes stands 4 (id - nodes) bytes behind the 8 nodes bytes of nodes
  const unsigned nodes = (1u << (depth - 1)) - 1u;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const unsigned l = w[k] + 4u * nodes + ((at[k] - w[k]) >> 1);
    leaf[k] = IN_LDS ? LdsAt<float>(l) : *reinterpret_cast<const float *>(words + l);
  }
}

// What bounds it: reads of the LDS, a node (8 bytes) and a value (4) per level, tree and row.  A
// workgroup owns R rows and holds all their values feature-major, so the 64 rows of a wave read 64
// banks whatever features their nodes ask for; the trees pass through the rest of the LDS in chunks,
// the next one fetched into registers while one is walked.  R is 1024 when there are rows enough to
// fill the chip: each staged tree then serves 1024 rows.  With fewer rows or more features R is
// smaller and the 1024 / R slices of the workgroup take different trees; the leaf weights they find
// meet in the LDS and are added in tree order.
// Beyond 467 float features not even 64 rows have their values in the LDS: they are read from memory row by row, a line
// per row and level.  (200 trees of depth 8, rows kept on the device: 200,000 x 400 0.70 ms, 200,000 x 500 1.55, 100,000 x
// 1000 1.50; a walk over columns, which meet in a line on the top levels only, took 1.81, 1.88 and 1.62.)
// 1,000,003 rows x 28 features, 200 trees of depth 8: 575 us (2370 with the values read from memory and
// a tree at a time), of which the LDS is busy 210 and the vector units 270; 64 rows by 100 trees of
// depth 6: 13 us (86).
template <int SRC, bool TILE, bool TREES_IN_LDS>
__global__ void __launch_bounds__(kWalkThreads) k_predict(const Walk a) {
  typedef typename Values<SRC>::T T;
  extern __shared__ __align__(16) unsigned char smem[];
  T *tile = reinterpret_cast<T *>(smem);
  uint2 *s_words = reinterpret_cast<uint2 *>(smem + a.words_at);
  float *s_leaf = reinterpret_cast<float *>(smem + a.leaf_at);
  const unsigned R = 1u << a.rows_log, r = threadIdx.x & (R - 1);
  const unsigned slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> a.rows_log), S = kWalkThreads >> a.rows_log;
  const unsigned row0 = blockIdx.x * R;
  const unsigned row = min(row0 + r, a.n - 1);
  const bool live = row0 + r < a.n;

  auto offset = [&](unsigned t) { return a.tree_words ? t * a.tree_words : a.refs[t].off; };
  auto chunk_end = [&](unsigned t0) { return min(a.n_trees, t0 + a.per_chunk); };
  uint2 ahead[kAhead];
  auto fetch_ahead = [&](unsigned t0) {
    const unsigned b = offset(t0), e = offset(chunk_end(t0));
#pragma unroll
    for (unsigned k = 0; k < kAhead; ++k) {
      const unsigned i = b + k * kWalkThreads + threadIdx.x;
      if (i < e) ahead[k] = a.words[i];
    }
  };
  if (TREES_IN_LDS) fetch_ahead(0);

  if (TILE) {
    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (SRC == kQuadCols) {
      const uint32_t *q = static_cast<const uint32_t *>(a.base);
      for (unsigned f4 = 4 * slice; f4 < a.F; f4 += 4 * S) {
        const uint32_t v = q[(size_t)(f4 >> 2) * a.ld + row];
        for (unsigned c = 0; c < min(4u, a.F - f4); ++c) tile[(f4 + c) * R + r] = (unsigned char)(v >> (8 * c));
      }
    } else {
      // a wave takes 16 rows by 4 features at a time: its reads are runs of 4 values of each row (the
      // lines are used up within the workgroup), its writes meet 4 to a bank
      const T *x = static_cast<const T *>(a.base);
      const unsigned fours = (a.F + 3) / 4, all = (R / 16) * fours;
      for (unsigned g = wave; g < all; g += 4 * (kWalkThreads / 64)) {
        T v[4];
        unsigned at[4];
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
          const unsigned i = g + k * (kWalkThreads / 64);
          const unsigned rr = i / fours * 16 + (lane >> 2), f = i % fours * 4 + (lane & 3u);
          at[k] = f * R + rr;
          if (i < all && f < a.F) v[k] = x[(size_t)min(row0 + rr, a.n - 1) * a.F + f];
          else at[k] = ~0u;
        }
#pragma unroll
        for (unsigned k = 0; k < 4; ++k)
          if (at[k] != ~0u) tile[at[k]] = v[k];
      }
    }
  }
  if (TILE && !TREES_IN_LDS) __syncthreads();

  const Fetch<SRC, TILE> value{R * (unsigned)sizeof(T), LdsAddress(smem) + r * (unsigned)sizeof(T), a, row};
  unsigned cur = 0;
  float acc = a.init;
  auto add = [&](unsigned t, float w) {
    if (a.labels > 1) {
      const unsigned label = a.refs[t].label;
      while (cur != label) {
        if (live) a.out[(size_t)cur * a.out_ld + row] = acc;
        acc = a.init;
        ++cur;
      }
    }
    acc += w;
  };

  for (unsigned t0 = 0; t0 < a.n_trees; t0 = chunk_end(t0)) {
    const unsigned t1 = chunk_end(t0);
    const unsigned b = TREES_IN_LDS ? offset(t0) : 0u;
    if (TREES_IN_LDS) {
      const unsigned e = offset(t1);
      __syncthreads();  // the chunk before is no longer read
#pragma unroll
      for (unsigned k = 0; k < kAhead; ++k) {
        const unsigned i = k * kWalkThreads + threadIdx.x;
        if (b + i < e) s_words[i] = ahead[k];
      }
      for (unsigned i = kAhead * kWalkThreads + threadIdx.x; b + i < e; i += kWalkThreads) s_words[i] = a.words[b + i];
      __syncthreads();
      if (t1 < a.n_trees) fetch_ahead(t1);
    } else if (S > 1) {
      __syncthreads();  // the leaf weights of the chunk before have been added
    }
    const unsigned char *words = reinterpret_cast<const unsigned char *>(a.words);
    auto tree = [&](unsigned t) {
      return (unsigned)__builtin_amdgcn_readfirstlane((TREES_IN_LDS ? LdsAddress(smem) + a.words_at : 0u) + (offset(t) - b) * (unsigned)sizeof(uint2));
    };
    auto depth = [&](unsigned t) { return a.tree_words ? a.depth : a.refs[t].depth; };
    for (unsigned t = t0 + slice; t < t1;) {
      float leaf[kChains];
      const unsigned d = depth(t);
      bool four = t + (kChains - 1) * S < t1;
      for (unsigned k = 1; four && k < kChains; ++k) four = depth(t + k * S) == d;
      if (four) {
        unsigned w[kChains];
#pragma unroll
        for (unsigned k = 0; k < kChains; ++k) w[k] = tree(t + k * S);
        WalkTrees<TREES_IN_LDS>(words, w, d, value, leaf);
      } else {
        const unsigned w[1] = {tree(t)};
        WalkTrees<TREES_IN_LDS>(words, w, d, value, leaf);
      }
#pragma unroll
      for (unsigned k = 0; k < kChains; ++k) {
        if (k > 0 && !four) break;
        if (S == 1) add(t + k, leaf[k]);
        else s_leaf[(t + k * S - t0) * R + r] = leaf[k];
      }
      t += four ? kChains * S : S;
    }
    if (S > 1) {
      __syncthreads();
      if (slice == 0) {
        unsigned t = t0;
        for (; t + 8 <= t1; t += 8) {
          float w[8];
#pragma unroll
          for (unsigned k = 0; k < 8; ++k) w[k] = s_leaf[(t + k - t0) * R + r];
#pragma unroll
          for (unsigned k = 0; k < 8; ++k) add(t + k, w[k]);
        }
        for (; t < t1; ++t) add(t, s_leaf[(t - t0) * R + r]);
      }
    }
  }
  if (slice == 0 && live)
    for (; cur < a.labels; ++cur, acc = a.init) a.out[(size_t)cur * a.out_ld + row] = acc;
}

template <int SRC, bool TILE, bool TREES_IN_LDS>
void Launch(const Walk &a, size_t lds, hipStream_t stream) {
  static std::once_flag configured;
  std::call_once(configured, [] {
    HIP_OK(hipFuncSetAttribute((const void *)k_predict<SRC, TILE, TREES_IN_LDS>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWalkLds));
  });
  const unsigned R = 1u << a.rows_log;
  hipLaunchKernelGGL((k_predict<SRC, TILE, TREES_IN_LDS>), dim3((a.n + R - 1) / R), dim3(kWalkThreads), lds, stream, a);
  HIP_OK(hipGetLastError());
}

}  // namespace

// Keeps the model laid out on the device between calls, and the memory of the results.
struct DevicePredictor {
  hipStream_t stream = nullptr;
  unsigned *model = nullptr;  // refs, then words
  size_t model_bytes = 0, words_at = 0;
  // of which trees, for how many features and labels `model` is (the trees of a booster are only added to)
  size_t begin = 0, end = 0, features = 0, labels_of = 0;
  unsigned largest = 0, tree_words = 0, depth = 0;
  unsigned char *staged = nullptr;  // pinned
  size_t staged_bytes = 0;
  float *result = nullptr;  // pinned; the sums of the last call
  size_t result_floats = 0;

  ~DevicePredictor() {
    if (stream) (void)hipStreamSynchronize(stream);
    DevicePoolGive(model);
    PinnedPoolGive(staged);
    PinnedPoolGive(result);
    StreamPoolGive(stream);
  }

  void LayOut(const std::vector<RegTree> &trees, size_t b, size_t e, size_t F, size_t labels) {
    if (begin == b && end == e && features == F && labels_of == labels) return;
    end = begin = 0;
    // in order of labels (stable): the sums of one label are complete before the next one's start
    std::vector<unsigned> order;
    for (size_t k = 0; k < labels; ++k)
      for (size_t t = b; t < e; ++t)
        if (trees[t].label == k) order.push_back((unsigned)t);
    if (order.size() != e - b) throw std::runtime_error("tree label out of range");
    std::vector<TreeRef> refs;
    size_t words = 0;
    largest = tree_words = 0;
    depth = trees[b].depth;
    bool same = true;
    for (unsigned t : order) {
      const size_t w = TreeWords(trees[t]);
      refs.push_back(TreeRef{(unsigned)words, trees[t].depth, trees[t].label, 0u});
      words += w;
      if (words * sizeof(uint2) >= kMostModelBytes) throw std::runtime_error("model too large for device prediction");
      largest = std::max(largest, (unsigned)w);
      same = same && trees[t].depth == depth;
    }
    refs.push_back(TreeRef{(unsigned)words, 0u, 0u, 0u});
    if (same) tree_words = largest;
    words_at = refs.size() * sizeof(TreeRef);
    const size_t bytes = words_at + words * sizeof(uint2);
    if (bytes > model_bytes) {
      DevicePoolGive(model);
      model = nullptr;
      model_bytes = 0;
      model = static_cast<unsigned *>(DevicePoolTake(bytes));
      model_bytes = bytes;
    }
    // A small model (a round's trees) is copied from pinned memory behind nothing and waited for by
    // nobody: Run waits for the stream before it returns.
    const bool small = bytes <= ((size_t)256 << 10);
    if (small && bytes > staged_bytes) {
      PinnedPoolGive(staged);
      staged = nullptr;
      staged_bytes = 0;
      staged = static_cast<unsigned char *>(PinnedPoolTake(bytes));
      staged_bytes = bytes;
    }
    std::vector<unsigned char> large(small ? 0 : bytes);
    unsigned char *host = small ? staged : large.data();
    std::memcpy(host, refs.data(), words_at);
    unsigned char *at = host + words_at;
    for (unsigned t : order) {
      const RegTree &tr = trees[t];
      for (size_t k = 0; k < tr.fid.size(); ++k) {
        uint2 nd;
        float thr = tr.threshold[k];
        nd.x = tr.fid[k];
        if (tr.fid[k] >= F) {  // a feature the matrix does not have reads as NaN: always right
          nd.x = 0;
          thr = -std::numeric_limits<float>::infinity();
        }
        std::memcpy(&nd.y, &thr, sizeof(float));
        std::memcpy(at, &nd, sizeof(nd));
        at += sizeof(nd);
      }
      std::memcpy(at, tr.weights.data(), tr.weights.size() * sizeof(float));
      at += tr.weights.size() * sizeof(float);
    }
    if (small) HIP_OK(hipMemcpyAsync(model, host, bytes, hipMemcpyHostToDevice, stream));
    else CopyToDevice(model, host, bytes, stream);
    begin = b;
    end = e;
    features = F;
    labels_of = labels;
  }

  // rows [0, n) at `base` into out[label * out_ld + row]
  void Rows(int src, const void *base, size_t ld, size_t n, size_t F, size_t labels, float init, float *out,
            size_t out_ld) {
    Walk a;
    a.base = base;
    a.ld = ld;
    a.n = (unsigned)n;
    a.F = (unsigned)F;
    a.refs = reinterpret_cast<const TreeRef *>(model);
    a.words = reinterpret_cast<const uint2 *>(reinterpret_cast<const unsigned char *>(model) + words_at);
    a.n_trees = (unsigned)(end - begin);
    a.labels = (unsigned)labels;
    a.tree_words = tree_words;
    a.depth = depth;
    a.init = init;
    a.out = out;
    a.out_ld = out_ld;
    const size_t element = src == kFloatRows ? sizeof(float) : 1;
    const size_t tree_bytes = (size_t)largest * sizeof(uint2);
    auto tile_bytes = [&](unsigned log) { return ((F << log) * element + 15) / 16 * 16; };
    // As many rows as give a workgroup to every CU, and room for a good chunk of trees beside them.
    unsigned log = 10;
    while (log > 6 && (n >> log) < 256) --log;
    const size_t trees_want = tree_bytes > kWalkLds / 2 ? 0 : std::max(tree_bytes, kTreeLds);
    // (leaf weights found, per tree: eight trees at least)
    auto leaves = [](unsigned log) { return log < 10 ? (size_t)4 << log : (size_t)0; };
    while (log > 6 && tile_bytes(log) + trees_want + 8 * leaves(log) > kWalkLds) --log;
    const bool tile = tile_bytes(log) + trees_want + 8 * leaves(log) <= kWalkLds;
    size_t free_lds = kWalkLds - (tile ? tile_bytes(log) : 0);
    const size_t leaf_bytes = leaves(log);
    const bool trees_in_lds = tree_bytes + 8 * leaf_bytes <= free_lds;
    // (whole model at once where rows are few: every chunk ends with a sum that 15 waves wait for)
    if (log == 10) free_lds = std::min(free_lds, std::max(kTreeLds, tree_bytes));
    a.rows_log = log;
    a.words_at = tile ? (unsigned)tile_bytes(log) : 0u;
    size_t per = free_lds / ((trees_in_lds ? tree_bytes : 0) + std::max<size_t>(leaf_bytes, trees_in_lds ? 0 : 4));
    per = std::min<size_t>(std::max<size_t>(per, 1), a.n_trees);
    a.per_chunk = (unsigned)per;
    a.leaf_at = a.words_at + (unsigned)(trees_in_lds ? per * tree_bytes : 0);
    const size_t lds = a.leaf_at + per * leaf_bytes;
#define ARB_WALK(S)                                                    \
  do {                                                                 \
    if (tile && trees_in_lds) Launch<S, true, true>(a, lds, stream);   \
    else if (tile) Launch<S, true, false>(a, lds, stream);             \
    else if (trees_in_lds) Launch<S, false, true>(a, lds, stream);     \
    else Launch<S, false, false>(a, lds, stream);                      \
  } while (0)
    if (src == kFloatRows) ARB_WALK(kFloatRows);
    else if (src == kByteRows) ARB_WALK(kByteRows);
    else ARB_WALK(kQuadCols);
#undef ARB_WALK
  }

  const float *Run(const DataMatrix &data, const std::vector<RegTree> &trees, size_t first, size_t use, size_t labels,
                   float init, size_t row_begin, size_t row_end) {
    const size_t n = std::min(row_end, data.rows) - row_begin, F = data.columns_dense;
    if (n == 0 || F == 0) throw std::runtime_error("empty data matrix");
    // only the block-wise walk of a streamed matrix indexes rows with 64 bits
    const bool blocks = data.InBlocks();
    if (n >= (1ull << 31) && !blocks) throw std::runtime_error("too many rows");
    if (data.is_prebinned && data.prebinned.empty() && !blocks) throw std::runtime_error("pre-quantised matrix without bins");
    if (!stream) stream = StreamPoolTake();
    LayOut(trees, first, use, F, labels);
    // Kernels write the sums where the host reads them: stores of 256 bytes a wave, at the rate of a copy
    // and beside the walk.
    if (labels * n > result_floats) {
      PinnedPoolGive(result);
      result = nullptr;
      result_floats = 0;
      result = static_cast<float *>(PinnedPoolTake(labels * n * sizeof(float)));
      result_floats = labels * n;
    }
    // rows on the host: piece by piece through pinned memory into one device block (the stream keeps
    // a piece's copy behind the walk of the one before)
    auto through_block = [&](int src, const void *rows, size_t row_bytes) {
      const size_t piece = kStageBytes / row_bytes;
      if (piece == 0) throw std::runtime_error("too many features for device prediction");
      struct Block {
        void *p;
        ~Block() { DevicePoolGive(p); }  // (the staging has waited for the stream's copies, Run waits for its walks)
      };
      const size_t pieces = (n + piece - 1) / piece, group = std::max<size_t>(kBlockBytes / kStageBytes, 1);
      Block block{DevicePoolTake(group * piece * row_bytes)};
      auto rows_of = [&](size_t k) { return std::min(piece, n - k * piece); };
      StageToDevice(pieces, [&](size_t k) { return rows_of(k) * row_bytes; },
                    [&](size_t k, void *p) {
                      const char *from = static_cast<const char *>(rows) + k * piece * row_bytes;
                      ParallelFor(rows_of(k) * row_bytes, [&](size_t b, size_t e) {
                        std::memcpy(static_cast<char *>(p) + b, from + b, e - b);
                      }, (size_t)256 << 10);
                    },
                    [&](size_t k) { return static_cast<char *>(block.p) + k % group * piece * row_bytes; },
                    [&](size_t k) {
                      if (k % group != group - 1 && k != pieces - 1) return;
                      const size_t r0 = k / group * group * piece;
                      Rows(src, block.p, 0, std::min(group * piece, n - r0), F, labels, init, result + r0, n);
                    }, stream);
      HIP_OK(hipStreamSynchronize(stream));
    };
    if (!data.is_prebinned) {
      if (const float *rows = data.values->OnDevice()) Rows(kFloatRows, rows + row_begin * F, 0, n, F, labels, init, result, n);
      else through_block(kFloatRows, data.values->OnHost() + row_begin * F, F * sizeof(float));
    } else if (!blocks) {
      through_block(kByteRows, data.prebinned.data() + row_begin * F, F);
    } else {
      // streamed matrix: its pinned blocks of quad columns go up as they are
      const size_t br = data.stream_block_rows, Q = (F + 3) / 4;
      if (row_begin % br != 0) throw std::runtime_error("internal: a range of rows starts inside a block");
      void *block = DevicePoolTake(Q * br * sizeof(uint32_t));
      try {
        for (size_t b = 0; b * br < n; ++b) {
          const size_t r0 = b * br;
          HIP_OK(hipMemcpyAsync(block, data.stream_blocks[row_begin / br + b], Q * br * sizeof(uint32_t), hipMemcpyHostToDevice, stream));
          Rows(kQuadCols, block, br, std::min(br, n - r0), F, labels, init, result + r0, n);
        }
        HIP_OK(hipStreamSynchronize(stream));
      } catch (...) {
        (void)hipStreamSynchronize(stream);
        DevicePoolGive(block);
        throw;
      }
      DevicePoolGive(block);
    }
    HIP_OK(hipStreamSynchronize(stream));
    return result;
  }
};

DevicePredictor *CreateDevicePredictor() { return new DevicePredictor(); }
void FreeDevicePredictor(DevicePredictor *p) { delete p; }
const float *PredictOnDevice(DevicePredictor *p, const DataMatrix &data, const std::vector<RegTree> &trees,
                             size_t begin, size_t end, size_t labels, float init, size_t row_begin, size_t row_end) {
  return p->Run(data, trees, begin, end, labels, init, row_begin, row_end);
}

bool DeviceWalkFits(const DataMatrix &data, const std::vector<RegTree> &trees, size_t begin, size_t end) {
  size_t bytes = 0;
  for (size_t t = begin; t < end; ++t) bytes += TreeWords(trees[t]) * sizeof(uint2);
  if (bytes >= kMostModelBytes) return false;
  const size_t F = data.columns_dense;
  if (!data.is_prebinned) return F * sizeof(float) <= kStageBytes || data.values->OnDevice() != nullptr;
  return data.InBlocks() || F <= kStageBytes;
}

}  // namespace arb
