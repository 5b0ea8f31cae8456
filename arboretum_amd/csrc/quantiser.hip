// Quantile thresholds of feature columns on the GPU: a hand-written LSD radix
// sort of every column of a batch followed by the reference's threshold rule.
//
// Replaces cub::DeviceRadixSort::SortKeys + DeviceScan with the
// ValueSegmentIterator / ThresholdOutputIterator pair (src/io/io.cu:349-410,
// 27-153, 255-270):  with s = the sorted column and seg = max(1, n / hist_size),
// the k-th change of value (s[i] != s[i-1], NaN != NaN included) at position i
// writes its midpoint float((s[i] + s[i-1]) * 0.5) to slot
// min(k + 1, i / seg + 1) - 2, lowest midpoint wins; NaN midpoints are never
// stored.  NaNs of either sign sort last.
//
// Every kernel takes all columns of a batch (blockIdx.y): seventeen launches
// for a matrix, whatever its width.  Column by column, with a copy of the
// thresholds to the host after each, 10,000 rows x 28 features took 5.3 ms, all
// of it launches and waits.
#include <hip/hip_runtime.h>

#include <cmath>
#include <limits>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "memory_pool.h"
#include "quantiser.h"

namespace arb {
namespace {

#define HIP_OK(expr)                                                                        \
  do {                                                                                      \
    hipError_t e_ = (expr);                                                                 \
    if (e_ != hipSuccess)                                                                   \
      throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + " in " #expr); \
  } while (0)

constexpr int kSortThreads = 256;
constexpr int kSortRounds = 16;                          // keys per thread
constexpr int kSortTile = kSortThreads * kSortRounds;    // 4096 keys per workgroup
constexpr unsigned kNanKey = 0xffffffffu;

// Order-preserving map float -> uint32; every NaN maps to the largest key.
__device__ __forceinline__ unsigned KeyOf(float v) {
  if (v != v) return kNanKey;
  const unsigned b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float ValueOf(unsigned k) {
  if (k == kNanKey) return __uint_as_float(0x7fc00000u);
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// The first pass reads the column itself, the later ones keys.
template <bool FLOATS>
__device__ __forceinline__ unsigned LoadKey(const void *__restrict__ p, size_t i) {
  if (FLOATS) return KeyOf(static_cast<const float *>(p)[i]);
  return static_cast<const unsigned *>(p)[i];
}

// Digit counts of one tile: counts[digit * nblk + block] of the column's 256 * nblk.  grid (nblk, columns)
template <bool FLOATS>
__global__ void __launch_bounds__(kSortThreads)
k_rs_count(const void *__restrict__ in, size_t n, int shift, unsigned *__restrict__ counts, unsigned nblk) {
  __shared__ unsigned s_cnt[256];
  s_cnt[threadIdx.x] = 0;
  __syncthreads();
  const void *col = static_cast<const unsigned *>(in) + (size_t)blockIdx.y * n;
  const size_t base = (size_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int j = 0; j < kSortRounds; ++j) {
    const size_t i = base + (size_t)j * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&s_cnt[(LoadKey<FLOATS>(col, i) >> shift) & 255u], 1u);
  }
  __syncthreads();
  counts[((size_t)blockIdx.y * 256 + threadIdx.x) * nblk + blockIdx.x] = s_cnt[threadIdx.x];
}

// In-place exclusive scan of the `m` counters of a column, and its thresholds unset.  A workgroup per column.
__global__ void __launch_bounds__(1024)
k_rs_scan(unsigned *__restrict__ counters, size_t m, unsigned *__restrict__ thr, int hist_size) {
  __shared__ unsigned s_part[1024];
  unsigned *v = counters + (size_t)blockIdx.x * m;
  for (int i = threadIdx.x; i < hist_size; i += 1024) thr[(size_t)blockIdx.x * hist_size + i] = 0xff800000u;  // KeyOf(+INF)
  const size_t per = (m + 1023) / 1024;
  const size_t b = min(m, (size_t)threadIdx.x * per), e = min(m, b + per);
  unsigned sum = 0;
  for (size_t i = b; i < e; ++i) sum += v[i];
  s_part[threadIdx.x] = sum;
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    unsigned t[16], tot = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      t[k] = s_part[lane * 16 + k];
      tot += t[k];
    }
    unsigned incl = tot;
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned o = __shfl_up(incl, off);
      if (lane >= off) incl += o;
    }
    unsigned run = incl - tot;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      s_part[lane * 16 + k] = run;
      run += t[k];
    }
  }
  __syncthreads();
  unsigned run = s_part[threadIdx.x];
  for (size_t i = b; i < e; ++i) {
    const unsigned c = v[i];
    v[i] = run;
    run += c;
  }
}

// Exclusive scan of the tile counts of every digit: workgroup (d, column) scans that digit's nblk
// counts in place and writes the digit's total.
__global__ void __launch_bounds__(kSortThreads)
k_rs_scan_digits(unsigned *__restrict__ counts, unsigned nblk, unsigned *__restrict__ digit_total) {
  __shared__ unsigned s_wave[kSortThreads / 64];
  const size_t digit = (size_t)blockIdx.y * 256 + blockIdx.x;
  unsigned *v = counts + digit * nblk;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned carry = 0;
  for (unsigned base = 0; base < nblk; base += kSortThreads) {
    const unsigned i = base + threadIdx.x;
    const unsigned c = i < nblk ? v[i] : 0u;
    unsigned incl = c;
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned o = __shfl_up(incl, off);
      if (lane >= off) incl += o;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    unsigned before = carry;
#pragma unroll
    for (int w = 0; w < kSortThreads / 64; ++w) {
      if (w < wave) before += s_wave[w];
      carry += s_wave[w];
    }
    if (i < nblk) v[i] = before + incl - c;
    __syncthreads();
  }
  if (threadIdx.x == 0) digit_total[digit] = carry;
}

// Lanes of the wave holding the same 8-bit digit as this lane.
__device__ __forceinline__ unsigned long long DigitPeers(unsigned d, bool valid) {
  unsigned long long peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const unsigned long long m = __ballot((d >> b) & 1u);
    peers &= ((d >> b) & 1u) ? m : ~m;
  }
  return peers;
}

// Stable scatter of one tile by digit; offsets[digit * nblk + block] is the
// first output position of the tile's keys with that digit, less the keys of
// smaller digits.  The tile is put in order in the LDS first, so that the keys
// of a digit leave as one run; a wave numbers its 1024 keys alone (its own
// counter per digit), and the workgroup meets three times per tile.
template <bool FLOATS>
__global__ void __launch_bounds__(kSortThreads)
k_rs_scatter(const void *__restrict__ in, unsigned *__restrict__ out, size_t n, int shift,
             const unsigned *__restrict__ offsets, unsigned nblk,
             const unsigned *__restrict__ digit_total) {
  constexpr int kWaves = kSortThreads / 64;
  constexpr int kWaveKeys = kSortTile / kWaves;
  __shared__ unsigned s_keys[kSortTile];
  __shared__ unsigned s_wave[kWaves][256];  // keys of each digit of the wave; then where the wave's first one goes
  __shared__ unsigned s_first[256];         // place in the tile of the first key of each digit
  __shared__ unsigned s_out[256];           // output position of that key
  __shared__ unsigned s_tot[2][kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t column = blockIdx.y;
  const void *col = static_cast<const unsigned *>(in) + column * n;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) s_wave[w][threadIdx.x] = 0;
  const size_t base = (size_t)blockIdx.x * kSortTile;
  const unsigned held = (unsigned)min((size_t)kSortTile, n - base);
  unsigned key[kSortRounds], rank[kSortRounds];
#pragma unroll
  for (int j = 0; j < kSortRounds; ++j) {
    const unsigned i = wave * kWaveKeys + j * 64 + lane;
    key[j] = i < held ? LoadKey<FLOATS>(col, base + i) : 0u;
  }
  const unsigned total = digit_total[column * 256 + threadIdx.x];
  const unsigned offset = offsets[(column * 256 + threadIdx.x) * nblk + blockIdx.x];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortRounds; ++j) {
    const bool valid = wave * kWaveKeys + j * 64 + lane < held;
    const unsigned d = (key[j] >> shift) & 255u;
    const unsigned long long peers = DigitPeers(d, valid);
    const unsigned below = (unsigned)__popcll(peers & ((1ull << lane) - 1ull));
    const unsigned before = s_wave[wave][d];
    rank[j] = before + below;
    if (valid && below == 0) s_wave[wave][d] = before + (unsigned)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    // thread = digit: keys of smaller digits in the tile, and in the column
    unsigned mine = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const unsigned c = s_wave[w][threadIdx.x];
      s_wave[w][threadIdx.x] = mine;
      mine += c;
    }
    unsigned in_tile = mine, in_col = total;
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned a = __shfl_up(in_tile, off), b = __shfl_up(in_col, off);
      if (lane >= off) {
        in_tile += a;
        in_col += b;
      }
    }
    if (lane == 63) {
      s_tot[0][wave] = in_tile;
      s_tot[1][wave] = in_col;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
      in_tile += s_tot[0][w];
      in_col += s_tot[1][w];
    }
    s_first[threadIdx.x] = in_tile - mine;
    s_out[threadIdx.x] = in_col - total + offset;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortRounds; ++j) {
    const unsigned d = (key[j] >> shift) & 255u;
    if (wave * kWaveKeys + j * 64 + lane < held) s_keys[s_first[d] + s_wave[wave][d] + rank[j]] = key[j];
  }
  __syncthreads();
  unsigned *dst = out + column * n;
#pragma unroll
  for (int j = 0; j < kSortRounds; ++j) {
    const unsigned i = j * kSortThreads + threadIdx.x;
    if (i < held) {
      const unsigned k = s_keys[i], d = (k >> shift) & 255u;
      dst[s_out[d] + (i - s_first[d])] = k;
    }
  }
}

__device__ __forceinline__ bool IsBorder(const unsigned *__restrict__ keys, size_t i) {
  if (i == 0) return false;
  const float a = ValueOf(keys[i]), b = ValueOf(keys[i - 1]);
  return a != b;  // true for NaN; false for -0.0 against +0.0
}

// Changes of value per tile.
__global__ void __launch_bounds__(kSortThreads)
k_thr_count(const unsigned *__restrict__ sorted, size_t n, unsigned *__restrict__ counts) {
  const unsigned *keys = sorted + (size_t)blockIdx.y * n;
  __shared__ unsigned s_cnt[kSortThreads / 64];
  const size_t base = (size_t)blockIdx.x * kSortTile;
  unsigned c = 0;
  for (int j = 0; j < kSortRounds; ++j) {
    const size_t i = base + (size_t)j * kSortThreads + threadIdx.x;
    if (i < n && IsBorder(keys, i)) ++c;
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off);
  if ((threadIdx.x & 63) == 0) s_cnt[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned t = 0;
    for (int w = 0; w < kSortThreads / 64; ++w) t += s_cnt[w];
    counts[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = t;
  }
}

// Thresholds as ordered keys: thr[slot] = min over the changes mapped to slot.
// Every wave owns a contiguous quarter of the tile: it counts its changes,
// the workgroup synchronises once, then the wave numbers its changes alone.
__global__ void __launch_bounds__(kSortThreads)
k_thr_emit(const unsigned *__restrict__ sorted, size_t n, const unsigned *__restrict__ before, unsigned seg,
           int hist_size, unsigned *__restrict__ thresholds) {
  const unsigned *keys = sorted + (size_t)blockIdx.y * n;
  unsigned *thr = thresholds + (size_t)blockIdx.y * hist_size;
  constexpr int kWaves = kSortThreads / 64;
  constexpr int kWaveKeys = kSortTile / kWaves;
  __shared__ unsigned s_wave[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t wbase = (size_t)blockIdx.x * kSortTile + (size_t)wave * kWaveKeys;
  unsigned mine = 0;
  for (int j = 0; j < kWaveKeys; j += 64) {
    const size_t i = wbase + j + lane;
    mine += (unsigned)__popcll(__ballot(i < n && IsBorder(keys, i)));
  }
  if (lane == 0) s_wave[wave] = mine;
  __syncthreads();
  unsigned run = before[(size_t)blockIdx.y * gridDim.x + blockIdx.x];  // changes before this wave's keys
  for (int w = 0; w < wave; ++w) run += s_wave[w];
  for (int j = 0; j < kWaveKeys; j += 64) {
    const size_t i = wbase + j + lane;
    const bool border = i < n && IsBorder(keys, i);
    const unsigned long long m = __ballot(border);
    const unsigned long long below = m & ((1ull << lane) - 1ull);
    int slot = -3;
    float mid = 0.0f;
    if (border) {
      const unsigned k = run + (unsigned)__popcll(below) + 1u;  // inclusive count
      const float a = ValueOf(keys[i]), b = ValueOf(keys[i - 1]);
      mid = (float)((double)(float)(a + b) * 0.5);
      const unsigned long long pos_slot = (unsigned long long)(i / seg) + 1ull;
      slot = (int)((long long)min((unsigned long long)k + 1ull, pos_slot) - 2);
    }
    // Slots and midpoints grow with the position (NaN midpoints come last), so
    // the minimum of a slot is at its first change: only the first change of
    // each slot within the wave goes to memory.
    const int prev = below ? 63 - __clzll((long long)below) : lane;
    const int prev_slot = __shfl(slot, prev);
    const bool first = border && (below == 0ull || prev_slot != slot);
    if (first && mid == mid && slot >= 0 && slot < hist_size) {
      const unsigned mk = KeyOf(mid);
      if (mk < thr[slot]) atomicMin(&thr[slot], mk);
    }
    run += (unsigned)__popcll(m);
  }
}

// Thresholds as floats; the number of real bins (leading finite thresholds + 1, capped at hist_size:
// io.cu:403-410); whether the column has NaNs.  A workgroup per column.
__global__ void __launch_bounds__(256)
k_thr_finish(const unsigned *__restrict__ thr, float *__restrict__ out, int hist_size,
             const unsigned *__restrict__ sorted, size_t n, int *__restrict__ sizes, unsigned *__restrict__ has_nan) {
  __shared__ int s_unset;
  if (threadIdx.x == 0) s_unset = hist_size;
  __syncthreads();
  const size_t at = (size_t)blockIdx.x * hist_size;
  for (int i = threadIdx.x; i < hist_size; i += 256) {
    const float v = ValueOf(thr[at + i]);
    out[at + i] = v;
    if (isinf(v)) atomicMin(&s_unset, i);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    sizes[blockIdx.x] = min(s_unset + 1, hist_size);
    has_nan[blockIdx.x] = sorted[(size_t)blockIdx.x * n + n - 1] == kNanKey ? 1u : 0u;
  }
}

// Columns [f0, f0 + nf) of row-major rows -> columns of `ld` floats, from position `at` on.  Tiles of 64
// rows by up to 32 features through the LDS: both sides move runs.  grid (row tiles, feature tiles)
__global__ void __launch_bounds__(256)
k_rows_to_columns(const float *__restrict__ rows, size_t n, int F, int f0, int nf, float *__restrict__ out, size_t ld,
                  size_t at) {
  __shared__ float s[32 * 65];
  const size_t r0 = (size_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 32, w = min(32, nf - c0);
  const unsigned held = (unsigned)min((size_t)64, n - r0) * w;
  for (unsigned i = threadIdx.x; i < held; i += 256) {
    const unsigned r = i / w, f = i % w;
    s[f * 65 + r] = rows[(r0 + r) * F + f0 + c0 + f];
  }
  __syncthreads();
  for (unsigned i = threadIdx.x; i < 64u * w; i += 256) {
    const unsigned f = i >> 6, r = i & 63u;
    if (r0 + r < n) out[(size_t)(c0 + f) * ld + at + r0 + r] = s[f * 65 + r];
  }
}

}  // namespace

struct SortWorkspace {
  size_t n = 0;
  unsigned nblk = 0;
  int hist_size = 0;
  unsigned *keys[2] = {nullptr, nullptr};
  unsigned *counts = nullptr, *digit_total = nullptr, *thr = nullptr;
};

SortWorkspace *CreateSortWorkspace(size_t n, int hist_size, int columns) {
  std::unique_ptr<SortWorkspace, void (*)(SortWorkspace *)> ws(new SortWorkspace(), FreeSortWorkspace);
  ws->n = n;
  ws->hist_size = hist_size;
  ws->nblk = (unsigned)((n + kSortTile - 1) / kSortTile);
  auto take = [&](size_t words) { return static_cast<unsigned *>(DevicePoolTake(words * columns * sizeof(unsigned))); };
  ws->keys[0] = take(n);
  ws->keys[1] = take(n);
  ws->counts = take((size_t)256 * ws->nblk);
  ws->digit_total = take(256);
  ws->thr = take((size_t)hist_size);
  return ws.release();
}

void FreeSortWorkspace(SortWorkspace *ws) {
  if (!ws) return;
  void *p[] = {ws->keys[0], ws->keys[1], ws->counts, ws->digit_total, ws->thr};
  for (void *q : p)
    DevicePoolGive(q);
  delete ws;
}

void DeviceThresholds(SortWorkspace *ws, const float *d_cols, int columns, float *d_thr, int *d_sizes,
                      unsigned *d_has_nan, hipStream_t st) {
  const size_t n = ws->n;
  const unsigned nblk = ws->nblk;
  const int hs = ws->hist_size;
  const dim3 tiles(nblk, (unsigned)columns), threads(kSortThreads);
  const void *in = d_cols;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 8 * pass;
    unsigned *out = ws->keys[pass & 1];
    if (pass == 0) hipLaunchKernelGGL(k_rs_count<true>, tiles, threads, 0, st, in, n, shift, ws->counts, nblk);
    else hipLaunchKernelGGL(k_rs_count<false>, tiles, threads, 0, st, in, n, shift, ws->counts, nblk);
    hipLaunchKernelGGL(k_rs_scan_digits, dim3(256, (unsigned)columns), threads, 0, st, ws->counts, nblk, ws->digit_total);
    if (pass == 0)
      hipLaunchKernelGGL(k_rs_scatter<true>, tiles, threads, 0, st, in, out, n, shift, ws->counts, nblk, ws->digit_total);
    else
      hipLaunchKernelGGL(k_rs_scatter<false>, tiles, threads, 0, st, in, out, n, shift, ws->counts, nblk, ws->digit_total);
    in = out;
  }
  const unsigned *sorted = ws->keys[1];
  unsigned seg = (unsigned)(n / (size_t)hs);
  if (seg < 1) seg = 1;
  hipLaunchKernelGGL(k_thr_count, tiles, threads, 0, st, sorted, n, ws->counts);
  hipLaunchKernelGGL(k_rs_scan, dim3((unsigned)columns), dim3(1024), 0, st, ws->counts, (size_t)nblk, ws->thr, hs);
  hipLaunchKernelGGL(k_thr_emit, tiles, threads, 0, st, sorted, n, ws->counts, seg, hs, ws->thr);
  hipLaunchKernelGGL(k_thr_finish, dim3((unsigned)columns), dim3(256), 0, st, ws->thr, d_thr, hs, sorted, n, d_sizes,
                     d_has_nan);
  HIP_OK(hipGetLastError());
}

void RowsToColumns(const float *d_rows, size_t n, int F, int f0, int nf, float *d_cols, size_t ld, size_t at,
                   hipStream_t st) {
  hipLaunchKernelGGL(k_rows_to_columns, dim3((unsigned)((n + 63) / 64), (unsigned)((nf + 31) / 32)), dim3(256), 0, st,
                     d_rows, n, F, f0, nf, d_cols, ld, at);
  HIP_OK(hipGetLastError());
}

}  // namespace arb
