// Column sweep: the vector kernel that the default launch runs at low block
// fill.  Each stored value is one gather of a B-row segment and one fused
// multiply-add per column; no padded block arithmetic.
//
// Why it gives the MFMA kernels' bits.  v_mfma_f32_16x16x4_f32 accumulates
// its four products as a chain of fused multiply-adds in k order (measured
// bit for bit against fmaf on 25 million random results, denormals
// included), and a zero of A adds +-0, which changes no finite sum.  So the
// chain of fmaf over a row's stored values alone, blocks in ascending order
// and the columns of a block in the order 0 2 4 6 1 3 5 7 (spmm_stream's two
// k-steps), gives the same bits, but for the sign of a zero: a sum whose every
// product so far rounded to -0 (negative, under half the smallest denormal)
// stays -0 here, where a zero term of the block kernels may lift it to +0.  What
// differs is B's infinities and NaNs: the block kernels multiply them by A's
// zeros and so poison every row of a window whose blocks hold the column.  Each
// wave therefore checks the sums it stores, and a non-finite one raises a mark
// on which k_sweep_repair (below) recomputes the product with A's zeros in it.
//
// Why this order.  Every gathered segment comes through the L2, and what
// bounds the SpMM on matrices without block structure is the rate of L2
// misses (5.6-7.5 TB/s whatever the gathers' order within a row).  The hits
// can be raised: when the waves of an XCD walk B from its first rows to its
// last at the same pace, a segment that one of them brings in serves the
// others.  The more rows are in flight at a time, the more gathers share
// each pass over B, so the sums of all rows in flight live in LDS (8 rows of
// 32 or 64 columns per lane group: 1280 or 640 rows per CU), the entry stream
// is sorted by column phase first and row second, and the waves of a
// workgroup keep step with a barrier every fourth batch.  Within a phase a
// row's values are consecutive, so the sum stays in registers and goes to
// LDS once per row and phase.
//
// Layout (built on the device, k_sweep_* below).  A wave is LG lane groups
// of C / 4 lanes; each lane group owns one list of RL rows.  An entry is
// (B row | row slot << 24 | kSweepFirst | kSweepLast, value): First = the
// first value of a run (the row's values of one phase), Last = its last.
// Lists are padded to 8 entries with null entries (value 0, no flags).  The
// lists do not depend on C: a wave takes 8 (C = 32) or 4 (C = 64)
// neighbouring ones.
//
// Measured against the block kernels at their default knobs (one MI355X, us):
// 4096 x 4096, 20 per row, N = 64 kernel 22.9 -> 7.6;
// 100003 x 30011, 10 per row, N = 128 68.9 -> 43.3, 21 % of L2 requests miss.  On
// the large matrices that the phase sweep (srbcrs_phasesweep.hpp) has taken
// since: uniform 65536 x 65536, 16 per row, N = 512 264 -> 190; power-law graph
// of 232965 nodes and 11.7 M values, N = 256 1755 -> 1290; of 2^20 nodes and
// 34.6 M values, N = 512 11560 -> 10400; phases and the barrier gave the
// 232965-node graph 1430 -> 1290.  Rejected: pacing the waves of an XCD against
// a shared counter (its atomics cost more than the hits gained: 1430 -> 1660
// before any wave waits).
#pragma once
#include "srbcrs_merged.hpp"

namespace srbcrs {

constexpr uint32_t kSweepFirst = 0x80000000u;
constexpr uint32_t kSweepLast = 0x40000000u;
constexpr int kSweepSlotShift = 24;
constexpr int kSweepBatch = 8;   // entries per list and batch
constexpr int kSweepLongBatch = 32;   // entries per batch of a long row (lists of entries are padded for it)

struct SweepStream {
  const uint2* entries;
  const int* start;   // first entry of each list
  const int* nblk;    // batches of each list
  const int* wblk;    // batches of each wave: the most of its lists
  const int* dest;    // RL per list: output row, -1 none, -2 - r partial row r
  int n_waves;
  const int* lstart;   // long rows: first entry, batches of kSweepLongBatch, output row (as dest)
  const int* lnblk;
  const int* ldest;
  int n_long;
};

// A sum about to be stored: its place in the output (or a partial tile).
__device__ __forceinline__ float* sweep_out(int d, int col, int64_t ldc, float* __restrict__ Cout,
                                            float* __restrict__ partial) {
  return d >= 0 ? Cout + (int64_t)d * ldc + col : partial + (int64_t)(-2 - d) * ldc + col;
}
__device__ __forceinline__ bool non_finite(float x) {
  return (__builtin_bit_cast(uint32_t, x) & 0x7f800000u) == 0x7f800000u;
}

// The mark of a run's non-finite sums.  A run launched eagerly has a number
// (token) and shares the mark with the runs 256 before and after it: raised to
// its number or beyond, the run is repaired, so a later run's at most costs a
// pass more.  A run recorded into a graph (token 0) has a mark of its own,
// {raised, replays, this replay}, and numbers its replays on the device: the
// sweep writes this replay's number for the repair pass and the repair pass
// counts it, each reading only what the other one wrote.
__device__ __forceinline__ void mark_begin(unsigned long long token, unsigned long long* __restrict__ mark) {
  if (token == 0 && blockIdx.x == 0 && threadIdx.x == 0) mark[2] = mark[1] + 1;
}
__device__ __forceinline__ void mark_raise(unsigned long long token, unsigned long long* __restrict__ mark) {
  atomicMax(mark, token ? token : mark[1] + 1);
}
__device__ __forceinline__ bool mark_raised(unsigned long long token, unsigned long long* __restrict__ mark) {
  const unsigned long long run = token ? token : mark[2];
  if (token == 0 && blockIdx.x == 0 && threadIdx.x == 0) mark[1] = run;
  return mark[0] >= run;
}

// One long row, 64 columns (one per lane).
__device__ __forceinline__ void sweep_long_row(const SweepStream& s, int r, int chunk, const float* __restrict__ B,
                                               uint32_t b_bytes, float* __restrict__ Cout,
                                               float* __restrict__ partial, int N, uint32_t ldb4, int64_t ldc,
                                               int relu, unsigned long long token,
                                               unsigned long long* __restrict__ mark, int lane) {
  constexpr int U = kSweepLongBatch;
  const int nb = uniform_load(s.lnblk, r);
  const int col = chunk * 64 + lane;
  const uint32_t boff = (uint32_t)(col < N ? col : N - 1) * 4u;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)b_bytes, 0x00020000);
  const uint2* ep = s.entries + uniform_load(s.lstart, r);
  // lane l of a batch's first U lanes holds entry l; its B row is broadcast
  // through a scalar register into the load's scalar offset
  auto fetch = [&](int j) { return ep[(j < nb ? j : nb - 1) * U + (lane & (U - 1))]; };
  float b[2][U];
  auto issue = [&](float(&d)[U], uint2 m) {
    const uint32_t off = __umul24(m.x, ldb4);
#pragma unroll
    for (int q = 0; q < U; ++q)
      d[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           rs, boff, (int)__builtin_amdgcn_readlane((int)off, q), 0));
  };
  float acc = 0.f;
  auto add = [&](const float(&d)[U], uint2 m) {
#pragma unroll
    for (int q = 0; q < U; ++q)
      acc = __builtin_fmaf(__builtin_bit_cast(float, __builtin_amdgcn_readlane((int)m.y, q)), d[q], acc);
  };
  uint2 m0 = fetch(0), m1 = fetch(1), m2;
  issue(b[0], m0);
  __builtin_amdgcn_sched_barrier(0);
  for (int j = 0; j < nb; j += 2) {
    m2 = fetch(j + 2);
    issue(b[1], m1);
    __builtin_amdgcn_sched_barrier(0);
    add(b[0], m0);
    __builtin_amdgcn_sched_barrier(0);
    m0 = m2;
    m2 = fetch(j + 3);
    issue(b[0], m0);
    __builtin_amdgcn_sched_barrier(0);
    if (j + 1 < nb) add(b[1], m1);
    __builtin_amdgcn_sched_barrier(0);
    m1 = m2;
  }
  const int d = uniform_load(s.ldest, r);
  bool bad = false;
  if (d != -1 && col < N) {
    bad = non_finite(acc);
    if (relu && d >= 0) acc = relu1(acc);
    __builtin_nontemporal_store(acc, sweep_out(d, col, ldc, Cout, partial));
  }
  if (__any(bad) && lane == 0) mark_raise(token, mark);
}

// One workgroup = WV waves of LG lists on one chunk of C columns.
template <int C, int RL, int WV>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(WV == 1 ? 5 : 4))) void spmm_colsweep(
    SweepStream s, const float* __restrict__ B, uint32_t b_bytes, float* __restrict__ Cout,
    float* __restrict__ partial, int N, uint32_t ldb4, int64_t ldc, int n_chunks, int swept, int relu,
    unsigned long long token, unsigned long long* __restrict__ mark, int long_wgs) {
  mark_begin(token, mark);
  constexpr int LPG = C / 4, LG = 64 / LPG;
  __shared__ __attribute__((aligned(16))) float tile[WV * LG * RL * C];
  const int n_wg = (s.n_waves + WV - 1) / WV;
  const int bid = (int)blockIdx.x;
  const int wave = WV == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (bid < long_wgs) {   // whole workgroups: the barriers below are not theirs
    const int i = bid * WV + wave;
    if (i < s.n_long * ((N + 63) / 64))
      sweep_long_row(s, i % s.n_long, i / s.n_long, B, b_bytes, Cout, partial, N, ldb4, ldc, relu, token, mark, lane);
    return;
  }
  int wg, c;   // long_wgs is a multiple of the XCD count: XCD = id % 8 still
  sweep_chunk(bid - long_wgs, gridDim.x - long_wgs, n_wg, n_chunks, swept, wg, c);
  if (wg >= n_wg) return;
  const int grp = lane / LPG, sub = lane % LPG;
  int w = wg * WV + wave;
  const bool live = w < s.n_waves;
  if (!live) w = s.n_waves - 1;   // a wave past the last: no batches of its own, kept for the barriers
  const int list = w * LG + grp;
  int nb = 0;   // the workgroup's batches: all its waves run as many, for the barriers
#pragma unroll
  for (int i = 0; i < WV; ++i) {
    const int x = wg * WV + i < s.n_waves ? uniform_load(s.wblk, wg * WV + i) : 0;
    nb = x > nb ? x : nb;
  }
  f4* tile4 = reinterpret_cast<f4*>(tile) + wave * (LG * RL * C / 4);
#pragma unroll
  for (int i = 0; i < LG * RL * C / 256; ++i) tile4[i * 64 + lane] = f4{0.f, 0.f, 0.f, 0.f};
  const int col = c * C + 4 * sub;
  if (nb > 0) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)b_bytes, 0x00020000);
    const uint32_t boff = (uint32_t)(col < N - 4 ? col : N - 4) * 4u;   // columns past N: repeat the last (not stored)
    const int my = live ? s.nblk[list] : 0;
    const uint2* ep = s.entries + s.start[list] + (lane & 7);
    char* tb = reinterpret_cast<char*>(tile4) + grp * (RL * C * 4) + sub * 16;
    auto fetch = [&](int j) {
      const int k = j < my ? j : my - 1;
      uint2 m = ep[(k > 0 ? k : 0) * kSweepBatch];
      if (j >= my) {   // past the list's end: its last B rows again (cache hits), value 0, no flags
        m.x &= (1u << kSweepSlotShift) - 1u;
        m.y = 0u;
      }
      return m;
    };
    f4 b[2][kSweepBatch];
    auto issue = [&](f4(&d)[kSweepBatch], uint2 m) {
#define SRBCRS_ISSUE(q)                                                \
  d[q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128( \
                                    rs, __umul24(group_bcast<LPG, q>(m.x), ldb4) + boff, 0, 0))
      SRBCRS_ISSUE(0);
      SRBCRS_ISSUE(1);
      SRBCRS_ISSUE(2);
      SRBCRS_ISSUE(3);
      SRBCRS_ISSUE(4);
      SRBCRS_ISSUE(5);
      SRBCRS_ISSUE(6);
      SRBCRS_ISSUE(7);
#undef SRBCRS_ISSUE
    };
    f4 acc = f4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](uint32_t x, uint32_t vb, f4 bv) {
      const float v = __builtin_bit_cast(float, vb);
      f4* p = reinterpret_cast<f4*>(tb + ((x >> kSweepSlotShift) & 31u) * (C * 4));
      if (x & kSweepFirst) acc = *p;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(v, bv[e], acc[e]);
      if (x & kSweepLast) *p = acc;
    };
    auto add = [&](const f4(&d)[kSweepBatch], uint2 m) {
#define SRBCRS_STEP8(q) step(group_bcast<LPG, q>(m.x), group_bcast<LPG, q>(m.y), d[q])
      SRBCRS_STEP8(0);
      SRBCRS_STEP8(1);
      SRBCRS_STEP8(2);
      SRBCRS_STEP8(3);
      SRBCRS_STEP8(4);
      SRBCRS_STEP8(5);
      SRBCRS_STEP8(6);
      SRBCRS_STEP8(7);
#undef SRBCRS_STEP8
    };
    // a batch's gathers are issued a batch ahead of its sums, its entries a
    // batch ahead of its gathers; the sched_barriers keep that order
    uint2 m0 = fetch(0), m1 = fetch(1), m2;
    issue(b[0], m0);
    __builtin_amdgcn_sched_barrier(0);
    for (int j = 0; j < nb; j += 2) {
      // pacing only (no wave reads another's LDS): every fourth batch, twice
      // as often measured 3-7 % slower on uniform, never 10 % slower
      if (WV > 1 && (j & 2) == 0) __builtin_amdgcn_s_barrier();
      m2 = fetch(j + 2);
      issue(b[1], m1);
      __builtin_amdgcn_sched_barrier(0);
      add(b[0], m0);
      __builtin_amdgcn_sched_barrier(0);
      m0 = m2;
      m2 = fetch(j + 3);
      issue(b[0], m0);
      __builtin_amdgcn_sched_barrier(0);
      add(b[1], m1);
      __builtin_amdgcn_sched_barrier(0);
      m1 = m2;
    }
  }
  bool bad = false;
#pragma unroll
  for (int r = 0; r < RL; ++r) {
    const int d = s.dest[list * RL + r];
    f4 v = tile4[((grp * RL + r) * C) / 4 + sub];
    if (live && d != -1 && col < N) {
      bad = bad || non_finite(v[0]) || non_finite(v[1]) || non_finite(v[2]) || non_finite(v[3]);
      if (relu && d >= 0) v = relu4(v);
      __builtin_nontemporal_store(v, reinterpret_cast<f4*>(sweep_out(d, col, ldc, Cout, partial)));
    }
  }
  if (__any(bad) && lane == 0) mark_raise(token, mark);
}

// The tasks of the schedule whose partial sums the stream reproduces.
struct SweepTasks {
  const int* begin;    // blocks [begin[t], end[t])
  const int* end;
  const int* window;   // null: window t
  const int* slot;     // null: straight into the output
  int n;
};

// The product again with A's zeros in it, where the column sweep stored a
// non-finite value (its mark is raised): the block kernels' matrix
// instructions over all positions of the blocks, so the same infinities and
// NaNs.  A fixed grid of waves walks all (task, 64-column chunk) pairs; without
// the mark every one leaves at once.  A block's indices are fetched two blocks
// ahead, its values and B rows one ahead.
//
// Bound as the block kernels are (gathers' L2 misses); one MI355X, the pass
// alone: 65536 x 65536, 16 per row, N = 512 370 us (block kernels 275); 232965
// of 50, N = 256 2010; 8000 of 16, N = 128 17.  One multiply-add per position
// and column, its A values by scalar loads, took 1615, 8080 and 104.
static __global__ __launch_bounds__(64) void k_sweep_repair(unsigned long long* __restrict__ mark,
                                                            unsigned long long token, SweepTasks t,
                                                            const uint2* __restrict__ words,
                                                            const int* __restrict__ sidx,
                                                            const float* __restrict__ packed,
                                                            const float* __restrict__ B, float* __restrict__ C,
                                                            float* __restrict__ partial,
                                                            const int* __restrict__ rowmap, int M, int N,
                                                            int64_t ldb, int64_t ldc, int relu) {
  if (!mark_raised(token, mark)) return;
  const int n_chunks = (N + 63) / 64;
  const int j = threadIdx.x & 15, k = threadIdx.x >> 4;   // A: row j, column 2 k + step; B: 4 columns from 4 j
  for (int64_t i = blockIdx.x; i < (int64_t)t.n * n_chunks; i += gridDim.x) {
    const int task = (int)(i % t.n);
    const int col = (int)(i / t.n) * 64 + 4 * j;
    const float* Bc = B + (col < N ? col : N - 4);   // columns past N: the last again (not stored)
    const int64_t b0 = t.begin[task], b1 = t.end[task];
    f4 acc[4];   // [column of the 4][row of rows 4 k ..]
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = f4{0.f, 0.f, 0.f, 0.f};
    int2 ix = int2{0, 0};
    uint2 wd = uint2{0u, 0u};
    float a0 = 0.f, a1 = 0.f;
    f4 v0, v1;
    auto fetch = [&](int64_t b) {
      if (b >= b1) b = b1 - 1;
      ix = *reinterpret_cast<const int2*>(sidx + 8 * b + 2 * k);
      wd = words[4 * b + (j >> 2)];
    };
    auto load = [&] {
      v0 = *reinterpret_cast<const f4*>(Bc + (int64_t)ix.x * ldb);
      v1 = *reinterpret_cast<const f4*>(Bc + (int64_t)ix.y * ldb);
      const int bit = 8 * (j & 3) + 2 * k;
      const uint32_t n = wd.y + (uint32_t)__builtin_popcount(wd.x & ((1u << bit) - 1u)), own = (wd.x >> bit) & 3u;
      const float p0 = packed[n], p1 = packed[n + (own & 1u)];   // (zeros follow the stored values)
      a0 = (own & 1u) ? p0 : 0.f;
      a1 = (own & 2u) ? p1 : 0.f;
    };
    if (b0 < b1) {
      fetch(b0);
      load();
      fetch(b0 + 1);
    }
    for (int64_t b = b0; b < b1; ++b) {
      const f4 w0 = v0, w1 = v1;
      const float x0 = a0, x1 = a1;
      load();
      fetch(b + 2);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x0, w0[c], acc[c], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x1, w1[c], acc[c], 0, 0, 0);
    }
    const int slot = t.slot ? t.slot[task] : -1;
    if (col >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      f4 v = f4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
      if (slot >= 0) {
        *reinterpret_cast<f4*>(partial + ((int64_t)slot * 16 + 4 * k + r) * ldc + col) = v;
      } else {
        const int64_t row = (int64_t)(t.window ? t.window[task] : task) * 16 + 4 * k + r;
        if (relu) v = relu4(v);
        if (row < M) *reinterpret_cast<f4*>(C + (int64_t)(rowmap ? rowmap[row] : row) * ldc + col) = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Building the stream.

// See launch_window_spans.
static __global__ __launch_bounds__(256) void k_window_spans(const int* __restrict__ soff,
                                                             const int* __restrict__ sidx, int Mo,
                                                             unsigned long long* __restrict__ out) {
  unsigned long long span = 0, n = 0;
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < Mo; w += (int64_t)gridDim.x * 256) {
    const int64_t b0 = soff[w], b1 = soff[w + 1];
    if (b0 == b1) continue;
    span += (unsigned long long)(sidx[8 * b1 - 1] - sidx[8 * b0]) + 1;
    ++n;
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) {
    span += __shfl_xor(span, d);
    n += __shfl_xor(n, d);
  }
  if ((threadIdx.x & 63) == 0 && n) {
    atomicAdd(out, span);
    atomicAdd(out + 1, n);
  }
}

// Bins of row lengths: exact below 256, 8 per octave above.
constexpr int kSweepBins = 512;
__host__ __device__ inline int sweep_bin(int n) {
  if (n < 256) return n;
  const int o = 31 - __builtin_clz(n);   // 8..30
  return 256 + 8 * (o - 8) + ((n >> (o - 3)) & 7);
}
constexpr int kSweepRankRows = 16;   // rows per thread of k_sweep_rank

// The columns (bits 0..7) of block b in which task row r holds a value, and
// (extra) the columns that hold none in any row, which row 0 gathers with
// value 0 so that the block's every B row is looked at (an explicit +0 entry
// of the CSR; a window's padding columns repeat the one before).
__device__ __forceinline__ uint32_t sweep_bits(const uint2* __restrict__ words, const int* __restrict__ sidx,
                                               int64_t b, int r, uint2& word, uint32_t& extra) {
  const uint4* p = reinterpret_cast<const uint4*>(words + 4 * b);
  const uint4 lo = p[0], hi = p[1];
  word = r < 4 ? uint2{lo.x, lo.y} : r < 8 ? uint2{lo.z, lo.w} : r < 12 ? uint2{hi.x, hi.y} : uint2{hi.z, hi.w};
  extra = 0;
  if (r == 0) {
    uint32_t any = lo.x | lo.z | hi.x | hi.z;
    any |= any >> 16;
    any = (any | (any >> 8)) & 0xffu;
    if (any != 0xffu)
      for (int q = 0; q < 8; ++q)
        if (!((any >> q) & 1u) && (q == 0 || sidx[8 * b + q] != sidx[8 * b + q - 1])) extra |= 1u << q;
  }
  return (word.x >> (8 * (r & 3))) & 0xffu;
}

// Values of each task row, and their histogram.  8 lanes per row.
static __global__ __launch_bounds__(256) void k_sweep_len(SweepTasks t, const uint2* __restrict__ words,
                                                          const int* __restrict__ sidx, int* __restrict__ len,
                                                          int* __restrict__ hist) {
  __shared__ int h[kSweepBins];
  for (int i = threadIdx.x; i < kSweepBins; i += 256) h[i] = 0;
  __syncthreads();
  const int64_t rows = (int64_t)t.n * 16;
  const int sub = threadIdx.x & 7;
  for (int64_t v = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3); v < rows; v += (int64_t)gridDim.x * 32) {
    const int64_t b0 = t.begin[v >> 4], b1 = t.end[v >> 4];
    int n = 0;
    for (int64_t b = b0 + sub; b < b1; b += 8) {
      uint2 wd;
      uint32_t extra;
      const uint32_t own = sweep_bits(words, sidx, b, (int)(v & 15), wd, extra);
      n += __builtin_popcount(own | extra);
    }
    n += __shfl_xor(n, 1, 8);
    n += __shfl_xor(n, 2, 8);
    n += __shfl_xor(n, 4, 8);
    if (sub == 0) {
      len[v] = n;
      atomicAdd(&h[sweep_bin(n)], 1);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kSweepBins; i += 256)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// The rows of the bins from long_bin up are the long rows, in rank order.
// Deal the others, longest first, to the lists: round j gives every list its
// j-th row, in alternating direction, so that the lists' totals come out near
// each other and neighbouring lists (the lane groups of one wave) nearest.
static __global__ __launch_bounds__(256) void k_sweep_rank(SweepTasks t, const int* __restrict__ len,
                                                           const int* __restrict__ hist, int* __restrict__ used,
                                                           int n_lists, int RL, int long_bin,
                                                           const int* __restrict__ rowmap, int M,
                                                           int* __restrict__ vrow, int* __restrict__ dest,
                                                           int* __restrict__ list_len, int* __restrict__ lvrow,
                                                           int* __restrict__ ldest, int long_cap,
                                                           int* __restrict__ n_long) {
  __shared__ int base[kSweepBins], mine[kSweepBins], part[256], sh_longs;
  constexpr int PER = kSweepBins / 256;
  const int tid = threadIdx.x;
  int tot = 0;
  for (int i = 0; i < PER; ++i) tot += hist[kSweepBins - 1 - (tid * PER + i)];
  part[tid] = tot;
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {
    const int x = tid >= d ? part[tid - d] : 0;
    __syncthreads();
    part[tid] += x;
    __syncthreads();
  }
  int run = part[tid] - tot;   // rows in longer bins
  for (int i = 0; i < PER; ++i) {
    const int bin = kSweepBins - 1 - (tid * PER + i);
    base[bin] = run;
    run += hist[bin];
    mine[bin] = 0;
    if (bin == long_bin) sh_longs = run;   // rows in bins >= long_bin
  }
  __syncthreads();
  const int longs = sh_longs;
  if (blockIdx.x == 0 && tid == 0) *n_long = longs;
  const int64_t rows = (int64_t)t.n * 16;
  const int64_t r0 = (int64_t)blockIdx.x * (256 * kSweepRankRows);
  int bin[kSweepRankRows], at[kSweepRankRows];
#pragma unroll
  for (int i = 0; i < kSweepRankRows; ++i) {
    const int64_t v = r0 + i * 256 + tid;
    bin[i] = -1;
    if (v < rows) {
      const int n = len[v];
      bin[i] = sweep_bin(n);
      at[i] = atomicAdd(&mine[bin[i]], 1);
    }
  }
  __syncthreads();
  for (int i = tid; i < kSweepBins; i += 256)
    if (mine[i]) base[i] += atomicAdd(&used[i], mine[i]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSweepRankRows; ++i) {
    if (bin[i] < 0) continue;
    const int64_t v = r0 + i * 256 + tid;
    const int rank = base[bin[i]] + at[i];
    const int task = (int)(v >> 4), r = (int)(v & 15);
    const int slot = t.slot ? t.slot[task] : -1;
    int d;
    if (slot >= 0) {
      d = -2 - (slot * 16 + r);
    } else {
      const int64_t row = (int64_t)(t.window ? t.window[task] : task) * 16 + r;
      d = row < M ? (rowmap ? rowmap[row] : (int)row) : -1;
    }
    if (bin[i] >= long_bin) {
      if (rank < long_cap) {   // beyond it the build is given up
        lvrow[rank] = (int)v;
        ldest[rank] = d;
      }
    } else {
      const int k = rank - longs;
      const int j = k / n_lists, p = k % n_lists;
      const int list = (j & 1) ? n_lists - 1 - p : p;
      vrow[(int64_t)list * RL + j] = (int)v;
      dest[(int64_t)list * RL + j] = d;
      const int n = len[v];
      if (n) atomicAdd(&list_len[list], n);
    }
  }
}

// Room for the lists, 8 per thread (a wave's at C = 32, two waves' at 64);
// total[0] = entries taken.
static __global__ __launch_bounds__(64) void k_sweep_place(const int* __restrict__ list_len, int n8, int64_t cap,
                                                           int* __restrict__ start, int* __restrict__ nblk,
                                                           int* __restrict__ wblk8, int* __restrict__ wblk4,
                                                           unsigned long long* __restrict__ total) {
  const int w = blockIdx.x * 64 + threadIdx.x;
  int nb[8], sum = 0;
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    nb[g] = w < n8 ? (list_len[w * 8 + g] + kSweepBatch - 1) / kSweepBatch : 0;
    sum += nb[g];
  }
  int incl = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(incl, d);
    if ((int)threadIdx.x >= d) incl += x;
  }
  unsigned long long base = 0;
  if (threadIdx.x == 63) base = atomicAdd(total, (unsigned long long)incl * kSweepBatch);
  base = __shfl(base, 63);
  if (w >= n8) return;
  int64_t at = (int64_t)base + (int64_t)(incl - sum) * kSweepBatch;
  const bool fits = at + (int64_t)sum * kSweepBatch <= cap;
  int most[2] = {0, 0};
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    if (!fits) nb[g] = 0;
    start[w * 8 + g] = fits ? (int)at : 0;
    nblk[w * 8 + g] = nb[g];
    most[g / 4] = nb[g] > most[g / 4] ? nb[g] : most[g / 4];
    at += (int64_t)nb[g] * kSweepBatch;
  }
  wblk4[2 * w] = most[0];
  wblk4[2 * w + 1] = most[1];
  wblk8[w] = most[0] > most[1] ? most[0] : most[1];
}

// Room for the long rows, one per thread.
static __global__ __launch_bounds__(64) void k_sweep_place_long(const int* __restrict__ len,
                                                                const int* __restrict__ lvrow,
                                                                const int* __restrict__ n_long, int long_cap,
                                                                int64_t cap, int* __restrict__ lstart,
                                                                int* __restrict__ lnblk,
                                                                unsigned long long* __restrict__ total) {
  const int r = blockIdx.x * 64 + threadIdx.x;
  if (r >= *n_long || r >= long_cap) return;
  const int nb = (len[lvrow[r]] + kSweepLongBatch - 1) / kSweepLongBatch;
  const int64_t at = (int64_t)atomicAdd(total, (unsigned long long)nb * kSweepLongBatch);
  const bool fits = at + (int64_t)nb * kSweepLongBatch <= cap;
  lstart[r] = fits ? (int)at : 0;
  lnblk[r] = fits ? nb : 0;
}

// The entries of 8 rows (8 / RL lists) per wave, a row on 8 lanes: count its
// values by phase, then write each to its place.  A block's phase is that of
// its first column, so that the blocks of a row stay in order.
static __global__ __launch_bounds__(64) void k_sweep_fill(SweepTasks t, const uint2* __restrict__ words,
                                                          const int* __restrict__ sidx,
                                                          const float* __restrict__ packed,
                                                          const int* __restrict__ vrow, int64_t n_rows,
                                                          int rows_per_list, const int* __restrict__ list_len,
                                                          const int* __restrict__ start,
                                                          const int* __restrict__ nblk, int n_phases,
                                                          int phase_shift, const int* __restrict__ lvrow,
                                                          const int* __restrict__ len,
                                                          const int* __restrict__ lstart,
                                                          const int* __restrict__ lnblk,
                                                          const int* __restrict__ n_long, int long_cap,
                                                          uint2* __restrict__ entries) {
  const int lane = threadIdx.x, s8 = lane >> 3, sub = lane & 7;
  // workgroups past the lists' rows take 8 long rows each: lists of one row
  // and one phase
  const int64_t list_wgs = (n_rows + 7) / 8;
  const bool is_long = (int64_t)blockIdx.x >= list_wgs;
  const int RL = is_long ? 1 : rows_per_list, phases = is_long ? 1 : n_phases, shift = is_long ? 31 : phase_shift;
  const int unit = is_long ? kSweepLongBatch : kSweepBatch;
  const int64_t gl = ((int64_t)blockIdx.x - (is_long ? list_wgs : 0)) * 8 + s8;
  const int s = (int)(gl % RL), first8 = s8 - s;
  const int64_t list = gl / RL;
  const bool have = is_long ? gl < *n_long && gl < long_cap && lnblk[gl] > 0 : gl < n_rows && nblk[list] > 0;
  const int v = !have ? -1 : is_long ? lvrow[gl] : vrow[gl];
  extern __shared__ int sm[];
  int* cnt = sm;                  // [8][phases] values of the row in the phase
  int* off = sm + 8 * phases;     // [8][phases] place of the run in the list
  int* rank0 = sm + 16 * phases;  // [8][phases] rank in the row of the run's first value
  int* base = sm + 24 * phases;   // [8][phases] of each list: entries in earlier phases
  const int r = v & 15;
  int64_t b0 = 0, b1 = 0;
  if (v >= 0) {
    b0 = t.begin[v >> 4];
    b1 = t.end[v >> 4];
  }
  for (int i = lane; i < 8 * phases; i += 64) cnt[i] = 0;
  __syncthreads();
  for (int64_t b = b0 + sub; b < b1; b += 8) {
    uint2 wd;
    uint32_t extra;
    const uint32_t bits = sweep_bits(words, sidx, b, r, wd, extra) | extra;
    const int ph = sidx[8 * b] >> shift;
    if (bits) atomicAdd(&cnt[s8 * phases + ph], __builtin_popcount(bits));
  }
  __syncthreads();
  if (sub == 0) {
    int run = 0;
    for (int p = 0; p < phases; ++p) {
      rank0[s8 * phases + p] = run;
      run += cnt[s8 * phases + p];
    }
  }
  for (int p = sub; p < phases; p += 8) {
    int before = 0, all = 0;
    for (int q = 0; q < RL; ++q) {
      const int n = cnt[(first8 + q) * phases + p];
      if (q < s) before += n;
      all += n;
    }
    off[s8 * phases + p] = before;
    if (s == 0) base[s8 * phases + p] = all;
  }
  __syncthreads();
  if (sub == 0 && s == 0) {
    int run = 0;
    for (int p = 0; p < phases; ++p) {
      const int n = base[s8 * phases + p];
      base[s8 * phases + p] = run;
      run += n;
    }
  }
  __syncthreads();
  if (have) {
    uint2* out = entries + (is_long ? lstart[gl] : start[list]);
    int run = 0;
    for (int64_t bb = b0; bb < b1; bb += 8) {
      const int64_t b = bb + sub;
      uint2 wd = uint2{0u, 0u};
      uint32_t extra = 0, own = 0;
      if (b < b1) own = sweep_bits(words, sidx, b, r, wd, extra);
      const uint32_t bits = own | extra;
      const int n = __builtin_popcount(bits);
      int incl = n;
#pragma unroll
      for (int d = 1; d < 8; d <<= 1) {
        const int x = __shfl_up(incl, d, 8);
        if (sub >= d) incl += x;
      }
      if (n) {
        const int ph = sidx[8 * b] >> shift;
        const int lo = rank0[s8 * phases + ph], last = lo + cnt[s8 * phases + ph] - 1;
        int rank = run + incl - n;
        const int at = base[first8 * phases + ph] + off[s8 * phases + ph] - lo;
        for (int i = 0; i < 8; ++i) {
          const int q = ((2 * i) & 7) | (i >> 2);   // 0 2 4 6 1 3 5 7
          if (!((bits >> q) & 1u)) continue;
          const int bit = 8 * (r & 3) + q;
          const float val = ((own >> q) & 1u) ? packed[wd.y + __builtin_popcount(wd.x & ((1u << bit) - 1u))] : 0.f;
          const uint32_t x = (uint32_t)sidx[8 * b + q] | ((uint32_t)s << kSweepSlotShift) |
                             (rank == lo ? kSweepFirst : 0u) | (rank == last ? kSweepLast : 0u);
          out[at + rank] = uint2{x, __builtin_bit_cast(uint32_t, val)};
          ++rank;
        }
      }
      run += __shfl(incl, 7, 8);
    }
    const int have_n = is_long ? len[v] : list_len[list], room = (is_long ? lnblk[gl] : nblk[list]) * unit;
    if (s == 0)
      for (int i = have_n + sub; i < room; i += 8) out[i] = uint2{0u, 0u};
  }
}

}  // namespace srbcrs
