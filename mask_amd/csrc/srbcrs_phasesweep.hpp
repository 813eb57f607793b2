// Phase sweep: the column sweep (srbcrs_colsweep.hpp) with the rows of a
// workgroup pooled and every workgroup held to the same pace over B.
//
// The column sweep's lists advance through B entry by entry, and lists whose
// rows favour other columns drift apart: on a power-law graph of 232965 nodes
// the rows in flight on an XCD touch a tenth as many B rows as they have
// values, yet 58 % of the L2 requests missed.  Here B is cut into phases of
// equally many values.  A unit is two halves of up to 640 rows; a workgroup
// holds the sums of one half (16 waves at 64 columns, 8 at 32) or of both (16
// waves at 32) in LDS, and any lane group may add to any row of its half: per
// phase the rows' runs of values are dealt, longest first, to the half's 64
// lists, so that they come out within a value of each other, and a barrier
// ends the phase (the next one may give a row to another list).  Lists are
// padded to the phase's longest in whole batches (the null entries' gathers
// lie past B's end and fetch nothing); a mean of 13 values a list nearly always takes two, so all
// workgroups of the chip run the same number of batches in every phase and
// keep step without any of them waiting (means of 20 in three batches, 28 in
// four: 2-5 % slower on power-law graphs; means that spill over in some units:
// slower by more than the spill).  A row of more than 13 values in one phase
// would hold up the others: the rest of its run moves to the phases after it.
// Each row's values stay in order, so the bits are the column sweep's.
//
// The run's sum is read at its first value and written at its last; as runs
// follow each other on a list, both happen in one step.
//
// Measured against the column sweep (one MI355X, three B in turn, us): the
// 232965-node graph, N = 256 1284 -> 988 (misses 58 % -> 48 %), N = 128 666 ->
// 482; 2^20 nodes, 34.4 M values, N = 512 10570 -> 8680 (78 % -> 58 %); 116483 nodes, N = 256
// 292 -> 245; uniform 100000 x 100000, 30 per row, N = 256 276 -> 221; 65536 x
// 65536, 16 per row, N = 512 189 -> 182.
//
// What bounds it: with B small enough that every gather hits the L2, 475 us
// for the first graph's values at N = 256 (25 TB/s into the CUs), whatever the
// runs' lengths; above that the misses, and that a B row 1 or 2 KB from the
// next keeps to a few of the L2's channels (32 floats of padding gain 6-11 %,
// less than a padded copy of B costs).  Without effect: a third batch of
// gathers in flight; launches of a round or four each, which start the
// workgroups together (up to 5 % slower).  Slower: reading a batch's eight
// sums ahead of it (4-12 %).
#pragma once
#include "srbcrs_colsweep.hpp"

namespace srbcrs {

// Stream entry: kPhaseLast | row of the half << kPhaseRowShift | B row, value.
constexpr uint32_t kPhaseLast = 0x80000000u;
constexpr int kPhaseRowShift = 21;
constexpr uint32_t kPhaseNull = (1u << kPhaseRowShift) - 1u;   // B row of null entries, and the field's mask
constexpr int kPhaseMaxRows = 640;   // rows of a half; two halves of 32 columns fill 160 KB
constexpr int kPhaseLists = 128;     // lists of a unit
constexpr int kPhaseBins = 4096;     // of the column histogram
constexpr int kPhaseMax = 64;        // phases
constexpr int kPhaseLoad = 13;       // values per list and phase to aim at

struct PhaseStream {
  const uint2* entries;   // [batch][kPhaseLists][kSweepBatch], units one after the other
  const int* uoff;        // first batch of each unit, and the end
  const int* pend;        // [unit][phases]: batches of the unit up to the phase's end
  const int* dest;        // [half][rows]: output row, -1 none, -2 - r partial row r
  int n_units, phases, rows;
  SweepStream longs;      // the long rows
};

template <int C, int WV>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(4))) void spmm_phasesweep(
    PhaseStream s, const float* __restrict__ B, uint32_t b_bytes, float* __restrict__ Cout,
    float* __restrict__ partial, int N, uint32_t ldb4, int64_t ldc, int n_chunks, int swept, int relu,
    unsigned long long token, unsigned long long* __restrict__ mark, int n_ids) {
  mark_begin(token, mark);
  constexpr int LPG = C / 4, LG = 64 / LPG, SH = C == 32 ? 7 : 8, HALVES = WV * LG / 64;
  __shared__ __attribute__((aligned(16))) float tile[HALVES * kPhaseMaxRows * C];
  const int n_wg = s.n_units * (2 / HALVES);
  const int id = (int)blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (id >= n_ids) {   // whole workgroups: the barriers below are not theirs
    const int i = (id - n_ids) * WV + wave;
    if (i < s.longs.n_long * ((N + 63) / 64))
      sweep_long_row(s.longs, i % s.longs.n_long, i / s.longs.n_long, B, b_bytes, Cout, partial, N, ldb4, ldc, relu,
                     token, mark, lane);
    return;
  }
  int wg, c;
  sweep_chunk(id, n_ids, n_wg, n_chunks, swept, wg, c);
  if (wg >= n_wg) return;
  const int grp = lane / LPG, sub = lane % LPG;
  const int unit = HALVES == 2 ? wg : wg >> 1;
  const int rows = HALVES * s.rows;   // of this workgroup
  const int list = (HALVES == 2 ? 0 : (wg & 1) * 64) + wave * LG + grp;
  const uint32_t row0 = HALVES == 2 && wave >= WV / 2 ? (uint32_t)s.rows : 0u;
  f4* tile4 = reinterpret_cast<f4*>(tile);
  for (int i = threadIdx.x; i < rows * LPG; i += 64 * WV) tile4[i] = f4{0.f, 0.f, 0.f, 0.f};
  const int col = c * C + 4 * sub;
  const int u0 = uniform_load(s.uoff, unit), nb = uniform_load(s.uoff, unit + 1) - u0;
  auto barrier = [] {   // the sums are in LDS: only its operations are waited for
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  if (nb > 0) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)b_bytes, 0x00020000);
    const uint32_t boff = (uint32_t)(col < N - 4 ? col : N - 4) * 4u;   // columns past N: repeat the last (not stored)
    const uint2* ep = s.entries + ((int64_t)u0 * kPhaseLists + list) * kSweepBatch + (lane & 7);
    const int* pend = s.pend + (int64_t)unit * s.phases;
    auto fetch = [&](int j) { return ep[(int64_t)(j < nb ? j : nb - 1) * (kPhaseLists * kSweepBatch)]; };
    f4 b[2][kSweepBatch];
    auto issue = [&](f4(&d)[kSweepBatch], uint2 m) {
      const uint32_t row = m.x & kPhaseNull;
      // (with more than 4 KB of columns or B near 4 GB a null entry may land inside B: harmless)
      const uint32_t off = row == kPhaseNull ? 0u - 4096u : __umul24(row, ldb4);
#define SRBCRS_ISSUE(q)                                                \
  d[q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128( \
                                    rs, group_bcast<LPG, q>(off) + boff, 0, 0))
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
    uint32_t cur = kPhaseLast;   // the entry added last: flag and LDS offset of its row
    auto at = [&](uint32_t y) {
      return reinterpret_cast<f4*>(reinterpret_cast<char*>(tile) + ((y & 0x3ff80u) | (uint32_t)sub * 16u));
    };
    auto add = [&](const f4(&d)[kSweepBatch], uint2 m) {
      const uint32_t y = (m.x & kPhaseLast) | ((((m.x >> kPhaseRowShift) & 1023u) + row0) << SH);
      uint32_t next = group_bcast<LPG, 0>(y);
      if ((int)cur < 0) acc = *at(next);
#define SRBCRS_STEP(q, n)                                                                 \
  {                                                                                       \
    cur = next;                                                                           \
    const float v = __builtin_bit_cast(float, group_bcast<LPG, q>(m.y));                  \
    _Pragma("unroll") for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(v, d[q][e], acc[e]); \
    if (n < 8) next = group_bcast<LPG, n & 7>(y);                                         \
    if ((int)cur < 0) {                                                                   \
      *at(cur) = acc;                                                                     \
      if (n < 8) acc = *at(next);                                                         \
    }                                                                                     \
  }
      SRBCRS_STEP(0, 1);
      SRBCRS_STEP(1, 2);
      SRBCRS_STEP(2, 3);
      SRBCRS_STEP(3, 4);
      SRBCRS_STEP(4, 5);
      SRBCRS_STEP(5, 6);
      SRBCRS_STEP(6, 7);
      SRBCRS_STEP(7, 8);
#undef SRBCRS_STEP
    };
    int p = 0, end = 0;   // batches before `end` are of earlier phases or this one
    auto turn = [&](int j) {
      if (j < end) return;
      barrier();
      do end = uniform_load(pend, p++);
      while (end <= j);
      cur = kPhaseLast;
    };
    uint2 m0 = fetch(0), m1 = fetch(1), m2;
    issue(b[0], m0);
    __builtin_amdgcn_sched_barrier(0);
    for (int j = 0; j < nb; j += 2) {
      m2 = fetch(j + 2);
      issue(b[1], m1);
      __builtin_amdgcn_sched_barrier(0);
      turn(j);
      add(b[0], m0);
      __builtin_amdgcn_sched_barrier(0);
      m0 = m2;
      m2 = fetch(j + 3);
      issue(b[0], m0);
      __builtin_amdgcn_sched_barrier(0);
      if (j + 1 < nb) {
        turn(j + 1);
        add(b[1], m1);
      }
      __builtin_amdgcn_sched_barrier(0);
      m1 = m2;
    }
  }
  barrier();
  bool bad = false;
  const int* dest = s.dest + (int64_t)wg * rows;
  for (int r = wave * LG + grp; r < rows; r += WV * LG) {
    const int d = dest[r];
    f4 v = tile4[r * LPG + sub];
    if (d != -1 && col < N) {
      bad = bad || non_finite(v[0]) || non_finite(v[1]) || non_finite(v[2]) || non_finite(v[3]);
      if (relu && d >= 0) v = relu4(v);
      __builtin_nontemporal_store(v, reinterpret_cast<f4*>(sweep_out(d, col, ldc, Cout, partial)));
    }
  }
  if (__any(bad) && lane == 0) mark_raise(token, mark);
}

// ---------------------------------------------------------------------------
// Building the stream.

// Stored values by column (that of their block's first column).
static __global__ __launch_bounds__(256) void k_phase_hist(const uint2* __restrict__ words,
                                                           const int* __restrict__ sidx, int64_t n_blocks,
                                                           int bin_shift, int* __restrict__ hist) {
  __shared__ int h[kPhaseBins];
  for (int i = threadIdx.x; i < kPhaseBins; i += 256) h[i] = 0;
  __syncthreads();
  for (int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x; b < n_blocks; b += (int64_t)gridDim.x * 256) {
    const uint4* p = reinterpret_cast<const uint4*>(words + 4 * b);
    const uint4 lo = p[0], hi = p[1];
    atomicAdd(&h[sidx[8 * b] >> bin_shift], __builtin_popcount(lo.x) + __builtin_popcount(lo.z) +
                                                __builtin_popcount(hi.x) + __builtin_popcount(hi.z));
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kPhaseBins; i += 256)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// Bins to phases of about equally many values.
static __global__ __launch_bounds__(1024) void k_phase_cuts(const int* __restrict__ hist, int phases,
                                                            uint8_t* __restrict__ phase_of) {
  __shared__ unsigned long long part[1024];
  constexpr int PER = kPhaseBins / 1024;
  const int tid = threadIdx.x;
  unsigned long long sum = 0;
  for (int i = 0; i < PER; ++i) sum += (unsigned)hist[tid * PER + i];
  part[tid] = sum;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const unsigned long long x = tid >= d ? part[tid - d] : 0;
    __syncthreads();
    part[tid] += x;
    __syncthreads();
  }
  const unsigned long long total = part[1023] ? part[1023] : 1;
  unsigned long long before = part[tid] - sum;
  for (int i = 0; i < PER; ++i) {
    const unsigned n = (unsigned)hist[tid * PER + i];
    const unsigned long long p = (before + n / 2) * (unsigned)phases / total;
    phase_of[tid * PER + i] = (uint8_t)(p < (unsigned)phases ? p : phases - 1);
    before += n;
  }
}

// Values of each row of the halves by phase: cnt[half][phase][row].  A row on
// 8 lanes.  Where a row has more than `cap` in a phase (a row on one list is a
// chain) the rest moves to the next phases, and at the end back to earlier
// ones.
static __global__ __launch_bounds__(64) void k_phase_count(SweepTasks t, const uint2* __restrict__ words,
                                                           const int* __restrict__ sidx, const int* __restrict__ vrow,
                                                           int rows, int phases, int bin_shift, int cap,
                                                           const uint8_t* __restrict__ phase_of,
                                                           uint16_t* __restrict__ cnt) {
  __shared__ int n[8][kPhaseMax];
  const int lane = threadIdx.x, s8 = lane >> 3, sub = lane & 7;
  const int64_t slot = (int64_t)blockIdx.x * 8 + s8;
  const int64_t half = slot / rows;
  const int r = (int)(slot % rows);
  for (int i = lane; i < 8 * kPhaseMax; i += 64) n[0][i] = 0;
  __syncthreads();
  const int v = vrow[slot];
  if (v >= 0)
    for (int64_t b = t.begin[v >> 4] + sub; b < t.end[v >> 4]; b += 8) {
      uint2 wd;
      uint32_t extra;
      const uint32_t bits = sweep_bits(words, sidx, b, v & 15, wd, extra) | extra;
      if (bits) atomicAdd(&n[s8][phase_of[sidx[8 * b] >> bin_shift]], __builtin_popcount(bits));
    }
  __syncthreads();
  if (sub == 0) {
    int over = 0;
    for (int p = 0; p < phases; ++p) {
      const int x = n[s8][p] + over;
      over = x > cap && p + 1 < phases ? x - cap : 0;
      n[s8][p] = x - over;
    }
    for (int p = phases - 1; p > 0 && n[s8][p] > cap; --p) {
      n[s8][p - 1] += n[s8][p] - cap;
      n[s8][p] = cap;
    }
  }
  __syncthreads();
  for (int p = sub; p < phases; p += 8) cnt[(half * phases + p) * rows + r] = (uint16_t)n[s8][p];
}

// The runs (rows) of one half and phase to its 64 lists, longest first, in
// rounds of 16 to the 16 emptiest lists: place = entries before it << 6 | list.
constexpr int kPhaseRound = 16;
static __global__ __launch_bounds__(64) void k_phase_assign(const uint16_t* __restrict__ cnt, int rows,
                                                            uint32_t* __restrict__ place,
                                                            uint16_t* __restrict__ load, int* __restrict__ batches) {
  __shared__ int h[256];
  __shared__ uint32_t order[kPhaseMaxRows];   // length << 16 | row, longest first
  const int lane = threadIdx.x;
  const int64_t hp = blockIdx.x;
  for (int i = lane; i < 256; i += 64) h[i] = 0;
  __syncthreads();
  for (int r = lane; r < rows; r += 64) {
    const int n = cnt[hp * rows + r];
    atomicAdd(&h[255 - (n < 255 ? n : 255)], 1);
  }
  __syncthreads();
  int own[4], sum = 0;
  for (int i = 0; i < 4; ++i) {
    own[i] = h[lane * 4 + i];
    sum += own[i];
  }
  int at = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(at, d);
    if (lane >= d) at += x;
  }
  at -= sum;
  __syncthreads();
  for (int i = 0; i < 4; ++i) {
    h[lane * 4 + i] = at;
    at += own[i];
  }
  __syncthreads();
  for (int r = lane; r < rows; r += 64) {
    const int n = cnt[hp * rows + r];
    order[atomicAdd(&h[255 - (n < 255 ? n : 255)], 1)] = ((uint32_t)n << 16) | (uint32_t)r;
  }
  __syncthreads();
  uint32_t key = (uint32_t)lane;   // entries << 6 | list
  for (int i0 = 0; i0 < rows; i0 += kPhaseRound) {
    // ascending by entries
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        const uint32_t o = __shfl_xor(key, j);
        const bool up = (lane & k) == 0, lower = (lane & j) == 0;
        key = (up == lower) == (key < o) ? key : o;
      }
    const uint32_t x = lane < kPhaseRound && i0 + lane < rows ? order[i0 + lane] : 0u;
    const uint32_t n = x >> 16;
    if (__ballot(n != 0) == 0) break;
    if (n) {
      place[hp * rows + (x & 0xffffu)] = key;
      key += n << 6;
    }
  }
  load[hp * 64 + (key & 63u)] = (uint16_t)(key >> 6);
  int most = (int)(key >> 6);
#pragma unroll
  for (int d = 32; d; d >>= 1) most = max(most, __shfl_xor(most, d));
  if (lane == 0) batches[hp] = (most + kSweepBatch - 1) / kSweepBatch;
}

// Batches of a unit up to each phase's end (the longer half's), and the units'
// first batches; total[0] and [2] = their entries, [3] = their values.
static __global__ __launch_bounds__(1024) void k_phase_offsets(const int* __restrict__ batches,
                                                               const int* __restrict__ half_len, int n_units,
                                                               int phases, int* __restrict__ pend,
                                                               int* __restrict__ uoff,
                                                               unsigned long long* __restrict__ total) {
  __shared__ long long part[1024];
  const int tid = threadIdx.x;
  long long carry = 0;
  for (int u0 = 0; u0 < n_units; u0 += 1024) {
    const int u = u0 + tid;
    int n = 0;
    if (u < n_units)
      for (int p = 0; p < phases; ++p) {
        const int a = batches[(int64_t)(2 * u) * phases + p], b = batches[(int64_t)(2 * u + 1) * phases + p];
        n += a > b ? a : b;
        pend[(int64_t)u * phases + p] = n;
      }
    part[tid] = n;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
      const long long x = tid >= d ? part[tid - d] : 0;
      __syncthreads();
      part[tid] += x;
      __syncthreads();
    }
    if (u < n_units) {
      uoff[u] = (int)(carry + part[tid] - n);
      atomicAdd(total + 3, (unsigned long long)half_len[2 * u] + (unsigned long long)half_len[2 * u + 1]);
    }
    carry += part[1023];
    __syncthreads();
  }
  if (tid == 0) {
    uoff[n_units] = (int)carry;
    total[0] = total[2] = (unsigned long long)carry * (kPhaseLists * kSweepBatch);
  }
}

struct PhaseFill {
  const uint16_t* cnt;     // [half][phase][row]
  const uint32_t* place;
  const uint16_t* load;    // [half][phase][64]
  const int *uoff, *pend;
  int rows, phases;
};

// First entry of a list's batch: the list's entries are 8 in every batch.
__device__ __forceinline__ int64_t phase_entry(int64_t batch, int list, int i) {
  return ((batch + i / kSweepBatch) * kPhaseLists + list) * kSweepBatch + i % kSweepBatch;
}

// The entries of 8 rows per wave, a row on 8 lanes.
static __global__ __launch_bounds__(64) void k_phase_fill(SweepTasks t, const uint2* __restrict__ words,
                                                          const int* __restrict__ sidx,
                                                          const float* __restrict__ packed,
                                                          const int* __restrict__ vrow, PhaseFill f,
                                                          uint2* __restrict__ entries) {
  __shared__ int rank0[8][kPhaseMax], num[8][kPhaseMax], list[8][kPhaseMax], before[8][kPhaseMax];
  const int lane = threadIdx.x, s8 = lane >> 3, sub = lane & 7;
  const int64_t slot = (int64_t)blockIdx.x * 8 + s8;
  const int64_t half = slot / f.rows, unit = half >> 1;
  const int row = (int)(slot % f.rows);
  for (int p = sub; p < f.phases; p += 8) {
    const int64_t i = (half * f.phases + p) * f.rows + row;
    num[s8][p] = f.cnt[i];
    const uint32_t x = f.cnt[i] ? f.place[i] : 0u;
    list[s8][p] = (int)(x & 63u) + 64 * (int)(half & 1);
    before[s8][p] = (int)(x >> 6);
  }
  __syncthreads();
  if (sub == 0)
    for (int p = 0, run = 0; p < f.phases; ++p) {
      rank0[s8][p] = run;
      run += num[s8][p];
    }
  __syncthreads();
  const int v = vrow[slot];
  const int r = v & 15;
  const int64_t b0 = v >= 0 ? t.begin[v >> 4] : 0, b1 = v >= 0 ? t.end[v >> 4] : 0;
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
      int rank = run + incl - n, ph = 0;
      for (int i = 0; i < 8; ++i) {
        const int q = ((2 * i) & 7) | (i >> 2);   // 0 2 4 6 1 3 5 7
        if (!((bits >> q) & 1u)) continue;
        while (rank >= rank0[s8][ph] + num[s8][ph]) ++ph;
        const int bit = 8 * (r & 3) + q;
        const float val = ((own >> q) & 1u) ? packed[wd.y + __builtin_popcount(wd.x & ((1u << bit) - 1u))] : 0.f;
        const int64_t batch = (int64_t)f.uoff[unit] + (ph ? f.pend[unit * f.phases + ph - 1] : 0);
        const int i0 = rank - rank0[s8][ph];
        const uint32_t x = (uint32_t)sidx[8 * b + q] | ((uint32_t)row << kPhaseRowShift) |
                           (i0 + 1 == num[s8][ph] ? kPhaseLast : 0u);
        entries[phase_entry(batch, list[s8][ph], before[s8][ph] + i0)] = uint2{x, __builtin_bit_cast(uint32_t, val)};
        ++rank;
      }
    }
    run += __shfl(incl, 7, 8);
  }
}

// Null entries where a list's phase is shorter than its unit's: a B row past
// the end (the buffer load returns 0 and fetches nothing), value 0, never
// stored.
static __global__ __launch_bounds__(128) void k_phase_pad(PhaseFill f, uint2* __restrict__ entries) {
  const int64_t unit = blockIdx.x / f.phases;
  const int p = (int)(blockIdx.x % f.phases), list = threadIdx.x;
  const int begin = p ? f.pend[unit * f.phases + p - 1] : 0, end = f.pend[unit * f.phases + p];
  const int64_t batch = (int64_t)f.uoff[unit] + begin;
  const int n = f.load[((2 * unit + (list >> 6)) * f.phases + p) * 64 + (list & 63)];
  const int room = (end - begin) * kSweepBatch;
  if (n >= room) return;
  for (int i = n; i < room; ++i) entries[phase_entry(batch, list, i)] = uint2{kPhaseNull, 0u};
}

}  // namespace srbcrs
