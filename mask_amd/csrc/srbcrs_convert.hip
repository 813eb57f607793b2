// Device-side CSR -> SR-BCRS conversion (canonical preprocess_gpu rules),
// bit-exact with the host converter and with the reference's
// preprocess_gpu_srcfp32_srbcrs (examples/src_fp32/sr_bcrs/testbed/
// SRBCRSSpMM_kernel.cu:226-340): per BH-row window the sorted distinct
// columns, cut into BW-column blocks padded with the window's last column;
// values at the swizzled block offset, the last write winning for duplicate
// (row, column) pairs; edge_to_row / edge_to_col / block_partition; and the
// compact copy of the block values (srbcrs_compact.hip).
//
// A window's edges are contiguous in the CSR, so nothing needs a sort of the
// whole matrix: one workgroup sorts a window's (column, edge) keys in LDS,
// ranks the distinct columns and counts the stored values; a scan over the
// windows gives the block offsets; then 16 lanes (16x8) or a wave (32x32) per
// block write the block whole -- indices, mask words, stored values and the
// dense values, each byte once.  Every write has a single owner.
//
// Bound: the dense values, 512 bytes a block, written once (11.7 M edges of a
// power-law graph, 232965 rows, 1.4 M blocks: 0.71 GB of 0.95 GB moved, 190 us
// at the rate of a copy).  Measured on that graph (one MI355X): the windows 455
// us, blocks 382, scan 21 twice, of the 15 windows longer than LDS holds the keys
// and ranks 46 and the sort's 21 launches 130; the whole call 1.32 ms.  Sorting the whole matrix
// by (window, column, edge) with a device-wide sort, writing the blocks entry
// by entry over a fill, and copying the stored values out in a pass of their
// own took 43.5 ms; on 5000 rows with a product 535 us, now 203.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include <algorithm>

#include "srbcrs_convert.h"

namespace srbcrs {

namespace {

__device__ __forceinline__ int swz(int o) { return o ^ ((o & 0x60) >> 3); }

// What the host needs back before it can size the arrays, and the counters of
// the windows too long for one workgroup's LDS.
struct Head {
  unsigned long long totals;       // blocks | stored values << 32
  unsigned long long big_entries;
  int bad, negative;
  unsigned max_col1;               // largest column + 1 (all zero at the start)
  int n_list[2], n_big;            // windows listed for k_listed_windows<0 / 1>, and longer ones
};

// Per sorted entry (at its window's edge range): what the block pass reads.
struct Sorted {
  int* col;         // its column
  float* val;       // its value
  int* rank;        // rank of its column among the window's distinct ones
  int* stored;      // stored values of the window before it
  int* block;       // [e0 + j]: the window's first entry of block j
  uint8_t* row;     // row in the window, bit 7: the last of its (row, column) run
};

struct ConvArgs {
  const int* rowptr;
  const int* colind;
  const float* values;
  int num_nodes;
  int64_t nnz;
  int bh, bw;
  int *e2r, *e2c, *bp;   // e2c, bp may be null
  Sorted s;
  unsigned long long* wcount;   // per window: blocks | stored values << 32
  int *list[2], *big;           // windows of the longer classes
  Head* head;
};

// Entries of a window sorted in LDS: by 256, 512 and 1024 threads.
constexpr int kClass[3] = {2048, 4096, 16384};

__device__ __forceinline__ void note_max(unsigned* p, unsigned v) {
  if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}

// Row of edge e in a window whose row offsets are rp[0..rows].
__device__ __forceinline__ int row_of(const int* rp, int rows, int e) {
  int lo = 0, hi = rows;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (rp[mid] <= e) lo = mid; else hi = mid;
  }
  return lo;
}

// Inclusive scan over the workgroup; total in every thread.
template <int T>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* part, uint32_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  __syncthreads();
  if (lane == 63) part[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    if (w < wave) before += part[w];
    total += part[w];
  }
  return before + x;
}

// Stable sort of n <= T * IPT keys by their high word, of `bits` bits: radix
// passes of up to 8 bits, in LDS.  A wave owns a contiguous run of keys, so
// rank = keys of lower digits, of the same digit in earlier waves, and of the
// same digit before it in its wave (lanes with the digit found by ballots).
// The keys wait in registers while the counts are summed, so one copy in LDS
// is enough.  (A bitonic sort moved each key through LDS 55 to 105 times and
// was bound by that: on the graph above 960 us, the radix passes 460.)
template <int T, int IPT>
__device__ __forceinline__ void radix_sort(uint64_t* key, int n, int bits, uint32_t* hist, uint32_t* part) {
  constexpr int W = T / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  const int iters = (n + W * 64 - 1) / (W * 64);   // 64-key steps per wave
  const int first = wave * iters * 64 + lane;
  const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
  for (int shift = 0; shift < bits; shift += width) {
    const int digits = 1 << width;
    for (int i = threadIdx.x; i < digits * W; i += T) hist[i] = 0;
    __syncthreads();
    uint64_t k[IPT];
    uint32_t rank[IPT];
#pragma unroll
    for (int it = 0; it < IPT; ++it) {
      if (it < iters) {
        const int i = first + it * 64;
        const bool valid = i < n;
        k[it] = valid ? key[i] : 0;
        const uint32_t d = (uint32_t)(k[it] >> (32 + shift)) & (uint32_t)(digits - 1);
        uint64_t same = __ballot(valid);
        for (int b = 0; b < width; ++b) {
          const uint64_t ones = __ballot((d >> b) & 1u);
          same &= ((d >> b) & 1u) ? ones : ~ones;
        }
        // hist is digit-major: [digit][wave]
        const uint32_t before = valid ? hist[d * W + wave] : 0;
        rank[it] = before + (uint32_t)__popcll(same & below);
        __builtin_amdgcn_wave_barrier();
        if (valid && (same & below) == 0) hist[d * W + wave] = before + (uint32_t)__popcll(same);
        __builtin_amdgcn_wave_barrier();
      }
    }
    __syncthreads();
    // exclusive sums in (digit, wave) order
    const int per = digits * W / T > 0 ? digits * W / T : 1;
    uint32_t sum = 0, total;
    const int e0 = threadIdx.x * per;
    for (int e = e0; e < e0 + per && e < digits * W; ++e) sum += hist[e];
    uint32_t at = block_scan<T>(sum, part, total) - sum;
    for (int e = e0; e < e0 + per && e < digits * W; ++e) {
      const uint32_t c = hist[e];
      hist[e] = at;
      at += c;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IPT; ++it) {
      if (it < iters && first + it * 64 < n) {
        const uint32_t d = (uint32_t)(k[it] >> (32 + shift)) & (uint32_t)(digits - 1);
        key[hist[d * W + wave] + rank[it]] = k[it];
      }
    }
    __syncthreads();
  }
}

// Sorted entry i of a window: col(i) / edge(i).  flag: bit 0 the first of its
// column, bit 16 a stored value.
struct Entry {
  int c, e, row;
  float v;
  bool last;   // of its (row, column) run
  uint32_t flag;
};
template <class Col, class Edge>
__device__ __forceinline__ Entry entry_at(const ConvArgs& a, const int* rp, int rows, int n, int i, Col col,
                                          Edge edge) {
  Entry x;
  x.c = col(i);
  x.e = edge(i);
  x.row = row_of(rp, rows, x.e);
  const bool first = i == 0 || col(i - 1) != x.c;
  x.last = i + 1 == n || col(i + 1) != x.c || row_of(rp, rows, edge(i + 1)) != x.row;
  x.v = a.values[x.e];
  x.flag = (first ? 1u : 0u) | (x.last && __float_as_uint(x.v) != 0u ? 1u << 16 : 0u);
  return x;
}

// Tile of sorted keys -> ranks, stored counts and the per-entry outputs; firsts
// and stored carry the window's counts over the tiles before this one.
template <int T, class Col, class Edge>
__device__ __forceinline__ void rank_tile(const ConvArgs& a, const int* rp, int rows, int n, int i0,
                                          uint32_t& firsts, uint32_t& stored, uint32_t* part, Col col, Edge edge) {
  const int e0 = rp[0];
  const int i = i0 + (int)threadIdx.x;
  Entry x{0, 0, 0, 0.f, false, 0u};
  if (i < n) x = entry_at(a, rp, rows, n, i, col, edge);
  uint32_t total;
  const uint32_t incl = block_scan<T>(x.flag, part, total);
  if (i < n) {
    const int p = (int)(firsts + (incl & 0xffffu)) - 1;
    const int64_t at = (int64_t)e0 + i;
    a.s.col[at] = x.c;
    a.s.val[at] = x.v;
    a.s.rank[at] = p;
    a.s.stored[at] = (int)(stored + ((incl - x.flag) >> 16));
    a.s.row[at] = (uint8_t)(x.row | (x.last ? 0x80 : 0));
    if ((x.flag & 1u) && p % a.bw == 0) a.s.block[(int64_t)e0 + p / a.bw] = i;
    if (a.e2c) a.e2c[x.e] = p;
  }
  firsts += total & 0xffffu;
  stored += total >> 16;
}

__device__ __forceinline__ void put_count(const ConvArgs& a, int w, uint32_t firsts, uint32_t stored) {
  const uint32_t nb = (firsts + (uint32_t)a.bw - 1) / (uint32_t)a.bw;
  a.wcount[w] = (unsigned long long)nb | ((unsigned long long)stored << 32);
  if (a.bp) a.bp[w] = (int)nb;
}

// The window's row offsets into LDS; false (and head->bad) if they are not
// non-decreasing within [0, nnz].  Nothing of such a window is read.
__device__ __forceinline__ bool window_rows(const ConvArgs& a, int w, int* rp, int& rows) {
  const int64_t r0 = (int64_t)w * a.bh;
  rows = (int)(r0 + a.bh < a.num_nodes ? a.bh : a.num_nodes - r0);
  __syncthreads();   // rp may still be read for the workgroup's previous window
  bool bad = false;
  if ((int)threadIdx.x <= rows) {
    const int v = a.rowptr[r0 + threadIdx.x];
    rp[threadIdx.x] = v;
    bad = v < 0 || v > a.nnz || ((int)threadIdx.x < rows && a.rowptr[r0 + threadIdx.x + 1] < v);
  }
  if (__syncthreads_or(bad)) {
    if (threadIdx.x == 0) {
      a.head->bad = 1;   // every writer writes the same value
      a.wcount[w] = 0;
    }
    return false;
  }
  return true;
}

// Sort and rank one window of n <= T * IPT entries.
template <int T, int IPT>
__device__ __forceinline__ void sort_window(const ConvArgs& a, int w, const int* rp, int rows, int n, uint64_t* key,
                                            uint32_t* hist, uint32_t* part, int* most) {
  const int e0 = rp[0];
  if (threadIdx.x == 0) *most = 0;
  __syncthreads();
  int mx = 0;
  for (int i = threadIdx.x; i < n; i += T) {
    const int c = a.colind[e0 + i];
    mx = max(mx, c < 0 ? INT32_MAX : c);   // a negative column sorts past the others
    if (c < 0) a.head->negative = 1;
    key[i] = ((uint64_t)(uint32_t)c << 32) | (uint32_t)i;
    a.e2r[e0 + i] = w * a.bh + row_of(rp, rows, e0 + i);
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) mx = max(mx, __shfl_xor(mx, d));
  if ((threadIdx.x & 63) == 0) atomicMax(most, mx);
  __syncthreads();
  radix_sort<T, IPT>(key, n, 32 - __builtin_clz(*most | 1), hist, part);
  uint32_t firsts = 0, stored = 0;
  for (int i0 = 0; i0 < n; i0 += T)
    rank_tile<T>(a, rp, rows, n, i0, firsts, stored, part, [&](int i) { return (int)(key[i] >> 32); },
                 [&](int i) { return e0 + (int)(uint32_t)key[i]; });
  if (threadIdx.x == 0) {
    put_count(a, w, firsts, stored);
    note_max(&a.head->max_col1, (unsigned)*most + 1u);
  }
}

// One window per workgroup; the longer ones are listed for the other passes.
__global__ __launch_bounds__(256) void k_windows(ConvArgs a) {
  __shared__ uint64_t key[kClass[0]];
  __shared__ uint32_t hist[256 * 4], part[4];
  __shared__ int rp[33], most;
  const int w = blockIdx.x;
  int rows;
  if (!window_rows(a, w, rp, rows)) return;
  const int n = rp[rows] - rp[0];
  if (n == 0) {
    if (threadIdx.x == 0) put_count(a, w, 0, 0);
  } else if (n <= kClass[0]) {
    sort_window<256, kClass[0] / 256>(a, w, rp, rows, n, key, hist, part, &most);
  } else if (threadIdx.x == 0) {
    a.wcount[w] = 0;
    if (n <= kClass[2]) {
      const int q = n <= kClass[1] ? 0 : 1;
      a.list[q][atomicAdd(&a.head->n_list[q], 1)] = w;
    } else {
      a.big[atomicAdd(&a.head->n_big, 1)] = w;
      atomicAdd(&a.head->big_entries, (unsigned long long)n);
    }
  }
}

template <int Q>
__global__ __launch_bounds__(Q ? 1024 : 512) void k_listed_windows(ConvArgs a) {
  constexpr int T = Q ? 1024 : 512, CAP = kClass[Q + 1];
  __shared__ uint64_t key[CAP];
  __shared__ uint32_t hist[256 * (T / 64)], part[T / 64];
  __shared__ int rp[33], most;
  for (int i = blockIdx.x; i < a.head->n_list[Q]; i += gridDim.x) {
    const int w = a.list[Q][i];
    int rows;
    if (!window_rows(a, w, rp, rows)) continue;
    sort_window<T, CAP / T>(a, w, rp, rows, rp[rows] - rp[0], key, hist, part, &most);
    __syncthreads();
  }
}

// First key of each of the longest windows in the concatenation of theirs.
__global__ __launch_bounds__(64) void k_big_offsets(ConvArgs a, int64_t* __restrict__ off) {
  const int lane = threadIdx.x, n_big = a.head->n_big;
  int64_t at = 0;
  for (int b0 = 0; b0 < n_big; b0 += 64) {
    const int b = b0 + lane;
    int64_t n = 0;
    if (b < n_big) {
      const int64_t r0 = (int64_t)a.big[b] * a.bh;
      n = a.rowptr[r0 + a.bh < a.num_nodes ? r0 + a.bh : a.num_nodes] - a.rowptr[r0];
    }
    int64_t incl = n;
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t x = __shfl_up(incl, d);
      if (lane >= d) incl += x;
    }
    if (b < n_big) off[b] = at + incl - n;
    at += __shfl(incl, 63);
  }
}

// Windows too long for LDS: (index in a.big << 32 | column) keys of all of
// them, one after the other, for one device-wide stable sort.  A row of the
// grid takes every kBigRows-th window; 1024 workgroups in all.
constexpr int kBigRows = 64;
__global__ __launch_bounds__(256) void k_big_keys(ConvArgs a, int n_big, const int64_t* __restrict__ off,
                                                  uint64_t* __restrict__ keys, int* __restrict__ edges) {
  for (int b = blockIdx.y; b < n_big; b += gridDim.y) {
    const int w = a.big[b];
    const int64_t r0 = (int64_t)w * a.bh;
    const int64_t r1 = r0 + a.bh < a.num_nodes ? r0 + a.bh : a.num_nodes;
    const int e0 = a.rowptr[r0], n = a.rowptr[r1] - e0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
      const int c = a.colind[e0 + i];
      if (c < 0) a.head->negative = 1;
      keys[off[b] + i] = ((uint64_t)(uint32_t)b << 32) | (uint32_t)c;
      edges[off[b] + i] = e0 + i;
      int lo = 0, hi = (int)(r1 - r0);
      while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (a.rowptr[r0 + mid] <= e0 + i) lo = mid; else hi = mid;
      }
      a.e2r[e0 + i] = (int)r0 + lo;
    }
  }
}

// The long windows' tiles of 1024 sorted keys over `segs` workgroups each: pass 0
// counts the firsts and stored values of a segment, pass 1 ranks it behind the
// segments before it.  (With one workgroup a window the conversion of one of 16 M
// entries took 60 ms, now 2.0; on the 15 of the graph above the pass took 102 us of
// 1.40 ms, now 39.)
template <int PASS>
__global__ __launch_bounds__(1024) void k_big_rank(ConvArgs a, int segs, const int64_t* __restrict__ off,
                                                   const uint64_t* __restrict__ keys, const int* __restrict__ edges,
                                                   unsigned long long* __restrict__ counts) {
  __shared__ uint32_t part[16];
  __shared__ uint32_t before[2];
  __shared__ int rp[33];
  const int b = (int)(blockIdx.x / (unsigned)segs), g = (int)(blockIdx.x % (unsigned)segs), w = a.big[b];
  unsigned long long* cnt = counts + (int64_t)b * segs;
  int rows;
  if (!window_rows(a, w, rp, rows)) return;
  const int n = rp[rows] - rp[0];
  const int tiles = (n + 1023) / 1024, per = (tiles + segs - 1) / segs;
  const int t0 = g * per, t1 = t0 + per < tiles ? t0 + per : tiles;
  const uint64_t* k = keys + off[b];
  const int* ed = edges + off[b];
  auto col = [&](int i) { return (int)(uint32_t)k[i]; };
  auto edge = [&](int i) { return ed[i]; };
  if (threadIdx.x < 2) before[threadIdx.x] = 0;
  __syncthreads();
  if constexpr (PASS == 0) {
    uint32_t firsts = 0, stored = 0;
    for (int64_t i = (int64_t)t0 * 1024 + threadIdx.x; i < (int64_t)t1 * 1024 && i < n; i += 1024) {
      const uint32_t flag = entry_at(a, rp, rows, n, (int)i, col, edge).flag;
      firsts += flag & 1u;
      stored += flag >> 16;
    }
    uint32_t all_firsts, all_stored;
    block_scan<1024>(firsts, part, all_firsts);
    block_scan<1024>(stored, part, all_stored);
    if (threadIdx.x == 0) cnt[g] = (unsigned long long)all_firsts | ((unsigned long long)all_stored << 32);
  } else {
    if (t0 >= t1) return;
    if ((int)threadIdx.x < g) {   // segs <= 256
      const unsigned long long c = cnt[threadIdx.x];
      atomicAdd(&before[0], (uint32_t)c);
      atomicAdd(&before[1], (uint32_t)(c >> 32));
    }
    __syncthreads();
    uint32_t firsts = before[0], stored = before[1];
    for (int t = t0; t < t1; ++t) rank_tile<1024>(a, rp, rows, n, t * 1024, firsts, stored, part, col, edge);
    if (threadIdx.x == 0 && t1 == tiles) {
      put_count(a, w, firsts, stored);
      note_max(&a.head->max_col1, (unsigned)(uint32_t)k[n - 1] + 1u);   // (negative columns refuse the matrix)
    }
  }
}

// Exclusive sums over the windows (one workgroup): block offsets and the
// index of each window's first stored value.  Also zeroes the edge maps of
// edges outside rows [0, num_nodes).
__global__ __launch_bounds__(1024) void k_window_scan(ConvArgs a, int Mo, int* __restrict__ soff,
                                                      unsigned* __restrict__ vbase) {
  __shared__ unsigned long long part[16];
  constexpr int PER = 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned long long carry = 0;
  for (int64_t base = 0; base < Mo; base += 1024 * PER) {
    unsigned long long v[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int64_t w = base + (int64_t)threadIdx.x * PER + i;
      v[i] = w < Mo ? a.wcount[w] : 0;
      sum += v[i];
    }
    unsigned long long x = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned long long y = __shfl_up(x, d);
      if (lane >= d) x += y;
    }
    __syncthreads();
    if (lane == 63) part[wave] = x;
    __syncthreads();
    unsigned long long at = carry + x - sum;
    for (int q = 0; q < 16; ++q) {
      if (q < wave) at += part[q];
      carry += part[q];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int64_t w = base + (int64_t)threadIdx.x * PER + i;
      if (w < Mo) {
        soff[w] = (int)(at & 0xffffffffu);
        vbase[w] = (unsigned)(at >> 32);
      }
      at += v[i];
    }
  }
  if (threadIdx.x == 0) {
    soff[Mo] = (int)(carry & 0xffffffffu);
    a.head->totals = carry;
  }
  if (!a.head->bad) {
    const int64_t lo = a.rowptr[0], hi = a.rowptr[a.num_nodes];
    for (int64_t e = threadIdx.x; e < lo + (a.nnz - hi); e += 1024) {
      const int64_t q = e < lo ? e : hi + (e - lo);
      a.e2r[q] = 0;
      if (a.e2c) a.e2c[q] = 0;
    }
  }
}

// The blocks: G lanes each, kBlockSteps * 256 / G per workgroup.  Entries of
// one block are contiguous in the sorted order; the lanes drop their values
// into an LDS copy of the block, which then goes out whole.  The workgroup
// finds the window of its first block by a 256-way search (two dependent
// loads; with a binary search per block, 14 of them, 1.4 M blocks took 574 us,
// now 381: 2.2 TB/s, the latency of the entries' loads).
constexpr int kBlockSteps = 4;
template <int BH, int BW, int G>
__global__ __launch_bounds__(256) void k_blocks(ConvArgs a, int Mo, const int* __restrict__ soff,
                                                const unsigned* __restrict__ vbase, int64_t n_blocks,
                                                int* __restrict__ sidx, float* __restrict__ val,
                                                uint2* __restrict__ words, float* __restrict__ packed) {
  constexpr int SIZE = BH * BW, WORDS = SIZE / 32, PER_WG = 256 / G, PER = SIZE / G;
  __shared__ __attribute__((aligned(16))) float tile[PER_WG][SIZE];
  __shared__ uint32_t mask[PER_WG][WORDS];
  __shared__ int cols[PER_WG][BW];
  __shared__ int off[257];   // soff from the first block's window on
  const int g = threadIdx.x / G, lane = threadIdx.x % G;
  const int64_t first = (int64_t)blockIdx.x * (PER_WG * kBlockSteps);
  int w0 = 0, len = Mo;   // last w with soff[w] <= first, in [w0, w0 + len)
  while (len > 1) {
    const int step = (len + 255) / 256, i = (int)threadIdx.x * step;
    const int hit = __syncthreads_count(i < len && soff[w0 + i] <= first) - 1;
    w0 += hit * step;
    len = len - hit * step < step ? len - hit * step : step;
  }
  for (int i = threadIdx.x; i < 257; i += 256) off[i] = soff[w0 + i < Mo ? w0 + i : Mo];
  __syncthreads();
  for (int stp = 0; stp < kBlockSteps; ++stp) {
    const int64_t b = first + stp * PER_WG + g;
    const bool have = b < n_blocks;
    int w = 0, s0 = 0, s1 = 0, p0 = 0;
    int64_t e0 = 0;
    if (have) {
      int lo = 0, hi = 256, so, sn;   // last w with soff[w] <= b: the window holding block b
      if (b < off[256] || w0 + 256 >= Mo) {
        while (hi - lo > 1) {
          const int mid = (lo + hi) / 2;
          if (off[mid] <= b) lo = mid; else hi = mid;
        }
        w = w0 + lo < Mo ? w0 + lo : Mo - 1;
      } else {   // many empty windows in between
        lo = w0 + 256;
        hi = Mo;
        while (hi - lo > 1) {
          const int mid = lo + (hi - lo) / 2;
          if (soff[mid] <= b) lo = mid; else hi = mid;
        }
        w = lo;
      }
      so = soff[w];
      sn = soff[w + 1];
      const int j = (int)(b - so);
      const int64_t r0 = (int64_t)w * BH, r1 = r0 + BH < a.num_nodes ? r0 + BH : a.num_nodes;
      e0 = a.rowptr[r0];
      p0 = j * BW;
      s0 = a.s.block[e0 + j];
      s1 = b + 1 < sn ? a.s.block[e0 + j + 1] : a.rowptr[r1] - (int)e0;
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) tile[g][q * G + lane] = 0.f;
    for (int q = lane; q < WORDS; q += G) mask[g][q] = 0;
    __syncthreads();
    for (int q = s0 + lane; q < s1; q += G) {
      const int c = a.s.rank[e0 + q] - p0;
      const uint8_t r = a.s.row[e0 + q];
      const float v = a.s.val[e0 + q];
      cols[g][c] = a.s.col[e0 + q];
      if (r & 0x80) {
        const int pos = BW * (r & 0x7f) + c;
        tile[g][swz(pos)] = v;
        if (__float_as_uint(v) != 0u) atomicOr(&mask[g][pos >> 5], 1u << (pos & 31));
      }
    }
    const int ncols = have ? a.s.rank[e0 + s1 - 1] - p0 + 1 : 0;
    __syncthreads();
    if (have) {
      for (int q = lane; q < BW; q += G) sidx[b * BW + q] = cols[g][q < ncols ? q : ncols - 1];
#pragma unroll
      for (int q = 0; q < PER / 4; ++q)
        reinterpret_cast<float4*>(val + b * SIZE)[q * G + lane] =
            reinterpret_cast<const float4*>(tile[g])[q * G + lane];
      if (words) {
        uint32_t base = vbase[w] + (uint32_t)a.s.stored[e0 + s0];
        // the lane's positions [lane * PER, lane * PER + PER) lie in one word (PER 8 or 16)
        const int wd = lane * PER / 32;
        for (int q = 0; q < wd; ++q) base += (uint32_t)__builtin_popcount(mask[g][q]);
        const uint32_t m = mask[g][wd];
        const int bit0 = lane * PER % 32;
        if (bit0 == 0) words[b * WORDS + wd] = uint2{m, base};
        uint32_t at = base + (uint32_t)__builtin_popcount(m & ((1u << bit0) - 1u));
#pragma unroll
        for (int q = 0; q < PER; ++q)
          if ((m >> (bit0 + q)) & 1u) packed[at++] = tile[g][swz(lane * PER + q)];
      }
    }
    __syncthreads();
  }
}

int bits_for(int64_t v) {
  int b = 0;
  while ((int64_t(1) << b) <= v) ++b;
  return b < 1 ? 1 : b;
}

// Allocations of one conversion: given back together, after the stream has
// finished with them.
struct Temps {
  DeviceAlloc alloc;
  DeviceFree dfree;
  void* ctx;
  hipStream_t st;
  void* p[24];
  int n = 0;
  bool waited = false, idle = false;
  template <class T>
  T* get(size_t count) {
    void* q = n < 24 ? alloc(ctx, (count ? count : 1) * sizeof(T)) : nullptr;
    if (q) p[n++] = q;
    return static_cast<T*>(q);
  }
  hipError_t wait() {
    const hipError_t e = hipStreamSynchronize(st);
    waited = true;
    idle = e == hipSuccess;
    return e;
  }
  ~Temps() {
    if (!waited) (void)wait();
    for (int i = 0; i < n; ++i) dfree(ctx, p[i], idle);
  }
};

}  // namespace

hipError_t device_convert(const DeviceConvertIn& in, DeviceConvertOut& out, DeviceAlloc alloc,
                          DeviceFree dfree, void* ctx, hipStream_t st) {
#define SRBCRS_TRY(x)                        \
  do {                                       \
    const hipError_t e_ = (x);               \
    if (e_ != hipSuccess) return e_;         \
  } while (0)
  const int bh = in.blk_h, bw = in.blk_w;
  const int Mo = (in.num_nodes + bh - 1) / bh;
  const size_t nnz = (size_t)in.nnz;
  out.Mo = Mo;
  out.total = 0;
  out.bad = 0;
  out.max_col = -1;
  Temps t{alloc, dfree, ctx, st};
  ConvArgs a{in.rowptr, in.colind, in.values, in.num_nodes, in.nnz, bh, bw, in.edge_to_row, in.edge_to_col,
             in.block_partition, {}, nullptr, {nullptr, nullptr}, nullptr, nullptr};
  a.s.col = t.get<int>(nnz);
  a.s.val = t.get<float>(nnz);
  a.s.rank = t.get<int>(nnz);
  a.s.stored = t.get<int>(nnz);
  a.s.block = t.get<int>(nnz);
  a.s.row = t.get<uint8_t>(nnz);
  a.wcount = t.get<unsigned long long>((size_t)Mo);
  a.list[0] = t.get<int>((size_t)Mo);
  a.list[1] = t.get<int>((size_t)Mo);
  a.big = t.get<int>((size_t)Mo);
  a.head = t.get<Head>(1);
  unsigned* vbase = t.get<unsigned>((size_t)Mo);
  if (!a.s.col || !a.s.val || !a.s.rank || !a.s.stored || !a.s.block || !a.s.row || !a.wcount || !a.list[0] ||
      !a.list[1] || !a.big || !a.head || !vbase)
    return hipErrorOutOfMemory;
  Head h{};
  SRBCRS_TRY(hipMemsetAsync(a.head, 0, sizeof(h), st));
  hipLaunchKernelGGL(k_windows, dim3((unsigned)Mo), dim3(256), 0, st, a);
  SRBCRS_TRY(hipGetLastError());
  // (a window longer than a class is impossible where the matrix has no more entries than that)
  if (in.nnz > kClass[0])
    hipLaunchKernelGGL(k_listed_windows<0>, dim3((unsigned)(Mo < 1024 ? Mo : 1024)), dim3(512), 0, st, a);
  SRBCRS_TRY(hipGetLastError());
  if (in.nnz > kClass[1])
    hipLaunchKernelGGL(k_listed_windows<1>, dim3((unsigned)(Mo < 256 ? Mo : 256)), dim3(1024), 0, st, a);
  SRBCRS_TRY(hipGetLastError());
  auto scan = [&]() -> hipError_t {
    hipLaunchKernelGGL(k_window_scan, dim3(1), dim3(1024), 0, st, a, Mo, out.soff, vbase);
    SRBCRS_TRY(hipGetLastError());
    SRBCRS_TRY(hipMemcpyAsync(&h, a.head, sizeof(h), hipMemcpyDeviceToHost, st));
    SRBCRS_TRY(hipMemcpyAsync(out.h_soff, out.soff, ((size_t)Mo + 1) * 4, hipMemcpyDeviceToHost, st));
    return hipStreamSynchronize(st);
  };
  SRBCRS_TRY(scan());
  if (h.n_big && !h.bad) {
    // windows too long for LDS: one stable device-wide sort of all of theirs
    const size_t n = (size_t)h.big_entries;
    uint64_t *k0 = t.get<uint64_t>(n), *k1 = t.get<uint64_t>(n);
    int *i0 = t.get<int>(n), *i1 = t.get<int>(n);
    int64_t* d_off = t.get<int64_t>((size_t)h.n_big);
    if (!k0 || !k1 || !i0 || !i1 || !d_off) return hipErrorOutOfMemory;
    hipLaunchKernelGGL(k_big_offsets, dim3(1), dim3(64), 0, st, a, d_off);
    SRBCRS_TRY(hipGetLastError());
    const int grid_y = h.n_big < kBigRows ? h.n_big : kBigRows, segs = std::max(1, std::min(256, 2048 / h.n_big));
    unsigned long long* counts = t.get<unsigned long long>((size_t)h.n_big * segs);
    if (!counts) return hipErrorOutOfMemory;
    hipLaunchKernelGGL(k_big_keys, dim3((unsigned)(1024 / grid_y), (unsigned)grid_y), dim3(256), 0, st, a, h.n_big,
                       d_off, k0, i0);
    SRBCRS_TRY(hipGetLastError());
    hipcub::DoubleBuffer<uint64_t> kb(k0, k1);
    hipcub::DoubleBuffer<int> ib(i0, i1);
    size_t bytes = 0;
    const int end_bit = 32 + bits_for(h.n_big);
    SRBCRS_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, kb, ib, (int)n, 0, end_bit, st));
    void* tmp = t.get<char>(bytes);
    if (!tmp) return hipErrorOutOfMemory;
    SRBCRS_TRY(hipcub::DeviceRadixSort::SortPairs(tmp, bytes, kb, ib, (int)n, 0, end_bit, st));
    const dim3 grid((unsigned)(h.n_big * segs));
    hipLaunchKernelGGL(k_big_rank<0>, grid, dim3(1024), 0, st, a, segs, d_off, kb.Current(), ib.Current(), counts);
    SRBCRS_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_big_rank<1>, grid, dim3(1024), 0, st, a, segs, d_off, kb.Current(), ib.Current(), counts);
    SRBCRS_TRY(hipGetLastError());
    SRBCRS_TRY(scan());
  }
  if (h.bad || h.negative) {
    out.bad = h.bad ? 1 : 2;
    return hipSuccess;
  }
  out.max_col = (int)(h.max_col1 - 1u);
  out.total = (int64_t)(h.totals & 0xffffffffu);
  const int64_t n_packed = (int64_t)(h.totals >> 32);
  const int64_t n_words = out.total * bh * bw / 32;
  auto need = [&](size_t n) { return alloc(ctx, (n ? n : 1) * 4); };
  out.sidx = (int*)need((size_t)out.total * bw);
  out.val = (float*)need((size_t)out.total * bh * bw);
  if (!out.sidx || !out.val) return hipErrorOutOfMemory;
  if (out.total == 0) return hipSuccess;
  // without room for the compact copy the plan keeps reading val
  out.compact.words = (uint2*)need(2 * (size_t)n_words);
  out.compact.packed = (float*)need((size_t)(n_packed + kPackedPad));
  if (!out.compact.words || !out.compact.packed) {
    if (out.compact.words) dfree(ctx, out.compact.words, true);
    if (out.compact.packed) dfree(ctx, out.compact.packed, true);
    out.compact = CompactOut{};
  } else {
    out.compact.n_packed = n_packed;
    SRBCRS_TRY(hipMemsetAsync(out.compact.packed + n_packed, 0, kPackedPad * 4, st));
  }
  if (bh == 16)
    hipLaunchKernelGGL((k_blocks<16, 8, 16>), dim3((unsigned)((out.total + 63) / 64)), dim3(256), 0, st, a, Mo,
                       out.soff, vbase, out.total, out.sidx, out.val, out.compact.words, out.compact.packed);
  else
    hipLaunchKernelGGL((k_blocks<32, 32, 64>), dim3((unsigned)((out.total + 15) / 16)), dim3(256), 0, st, a, Mo,
                       out.soff, vbase, out.total, out.sidx, out.val, out.compact.words, out.compact.packed);
  SRBCRS_TRY(hipGetLastError());
  return t.wait();
#undef SRBCRS_TRY
}

}  // namespace srbcrs
