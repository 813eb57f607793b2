// Column sweep (srbcrs_colsweep.hpp): launcher and the device-side build of
// its entry stream.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "srbcrs_colsweep.hpp"
#include "srbcrs_convert.h"
#include "srbcrs_kernels.h"
#include "srbcrs_phasesweep.hpp"

namespace srbcrs {

// Workgroups for sweep_chunk.
static int64_t sweep_grid(int64_t n_wg, int n_chunks, int swept) {
  if (swept || n_chunks > kNumXcd || kNumXcd % n_chunks) return n_wg * n_chunks;
  const int per = kNumXcd / n_chunks;
  return (n_wg + per - 1) / per * kNumXcd;
}

template <int C, int RL, int WV>
static hipError_t launch_t(const ColSweep& s, const StreamArgs& a, int64_t K, int swept, unsigned long long token,
                           unsigned long long* mark, hipStream_t st) {
  const int n_chunks = (a.N + C - 1) / C;
  const int n_waves = s.n_lists / (256 / C);
  const int64_t n_wg = (n_waves + WV - 1) / WV;
  int64_t grid = sweep_grid(n_wg, n_chunks, swept);
  const int64_t long_waves = (int64_t)s.n_long * ((a.N + 63) / 64);
  const int64_t long_wgs = ((long_waves + WV - 1) / WV + kNumXcd - 1) / kNumXcd * kNumXcd;
  grid += long_wgs;
  if (grid == 0) return hipSuccess;
  if (long_waves > INT32_MAX || grid > INT32_MAX) return hipErrorInvalidConfiguration;
  const uint64_t bytes = ((uint64_t)(K - 1) * (uint64_t)a.ldb + (uint64_t)a.N) * 4u;
  const SweepStream ss{s.entries, s.start, s.nblk, C == 32 ? s.wblk8 : s.wblk4, s.dest, n_waves,
                       s.lstart, s.lnblk, s.ldest, s.n_long};
  hipLaunchKernelGGL((spmm_colsweep<C, RL, WV>), dim3((unsigned)grid), dim3(64 * WV), 0, st, ss, a.B, (uint32_t)bytes,
                     a.C, a.partial, a.N, (uint32_t)(a.ldb * 4), a.ldc, n_chunks, swept, a.relu, token, mark,
                     (int)long_wgs);
  return hipGetLastError();
}

// Which kernel a launch runs, from sweeps of every (columns, waves per
// workgroup, mapping) over 17 matrices and widths 48-512 on one MI355X
// (fastest setting / the setting the rule would otherwise take, us).
//
// 64 columns where 32-column segments would straddle cache lines (N = 112,
// 100000 rows of 30: 143 / 157) or where the columns' 64-wide slice of B fits
// an XCD's L2 anyway (K = 8000, N = 256: 54 / 61); below 200000 rows also
// where the 32-column chunks are exactly 8, one per XCD: with B rows of 1 KB
// each XCD then sees one 128-byte phase of every KB, which its L2 channels do
// not spread (N = 256, 65536 rows: 85 / 92).  Else 32 columns: twice the rows
// in flight per CU (65536 rows of 16, N = 64: 29 / 32; power-law, 131072
// nodes, N = 512: 968 / 1045).
//
// A workgroup of 16 waves in step where B's slice exceeds the L2 (K = 100000,
// 30000 rows, N = 512: 104 / 137) and the workgroups fill their last round of
// CUs (one workgroup per CU): a round that is mostly empty costs more
// (power-law, 116483 nodes, N = 128, 1.8 rounds: 139 one wave / 165).  These
// launches are the phase sweep's unless it cannot take the matrix (more than
// 2^21 columns, or padding of half the values and more).
//
// Chunks are pinned to XCDs (an XCD's rows in flight are then all rows of its
// chunk) except for 32-column chunks of so many rows that one XCD's eighth of
// them fills it: then all XCDs take a chunk at the same time and share its B
// rows in the memory-side cache (524288 nodes, N = 256: 1820 / 1940).
constexpr int64_t kSyncBytes = 6 << 20;     // B slice above which waves keep step (4 MB of L2 hold the hot rows)
constexpr int64_t kSweptRows = 200000;
constexpr int64_t kMemCacheBytes = 256 << 20;

static void pick_launch(int64_t rows, int RL, const StreamArgs& a, int64_t K, int& cols, int& wv, int& swept) {
  const int64_t chunks32 = (a.N + 31) / 32;
  const bool sync = K * 128 > kSyncBytes;
  cols = a.N % 32 || a.ldb % 32 || K <= 16384 || (sync && chunks32 == kNumXcd && rows < kSweptRows) ? 64 : 32;
  const int64_t waves = rows / (8 * RL) * chunks32;
  const int64_t wgs = waves / 16, rounds = (wgs + 255) / 256;
  wv = sync && RL == 8 && waves >= 3500 && (rounds > 3 || 10 * wgs >= 9 * 256 * rounds) ? 16 : 1;
  swept = cols == 32 && rows >= kSweptRows;
}

hipError_t launch_window_spans(const int* soff, const int* sidx, int Mo, unsigned long long* out, hipStream_t st) {
  const int64_t g = ((int64_t)Mo + 255) / 256;
  if (g == 0) return hipSuccess;
  hipLaunchKernelGGL(k_window_spans, dim3((unsigned)(g < 1024 ? g : 1024)), dim3(256), 0, st, soff, sidx, Mo, out);
  return hipGetLastError();
}

int colsweep_rows_per_list(int64_t rows, int N) {
  const int64_t chunks32 = (N + 31) / 32;
  int RL = 8;
  while (RL > 1 && rows / (8 * RL) * chunks32 < 2000) RL /= 2;
  return RL;
}

// Where the phase sweep runs: B's 32-column slice exceeds an XCD's L2 by so
// much that phases pay (40000 rows of a power-law graph, K = 40000, N = 256:
// lists 152 us, phases 204; 58241: 226 / 214) and its workgroups, one per CU,
// fill three quarters of the chip (65536 rows of 16, N = 64, half of it: 24 /
// 30; N = 128: 46 / 41; power-law, 116483 nodes, N = 48: 77 / 72).
//
// Rows per half: as many as make the last round of workgroups a full one.
int phasesweep_rows(int64_t rows, int N, int64_t K) {
  const int64_t chunks = ((int64_t)N + 31) / 32;
  if (K * 128 <= kSyncBytes || K > (int64_t)kPhaseNull || rows / 64 * chunks < 3000) return 0;
  for (int64_t rounds = 1;; ++rounds) {
    const int64_t units = 256 * rounds / chunks;
    if (units == 0) continue;
    const int64_t r = (rows + 2 * units - 1) / (2 * units);
    if (r <= kPhaseMaxRows) return (int)((r + 7) / 8 * 8);
  }
}

template <int C, int WV>
static hipError_t launch_phase_t(const ColSweep& s, const StreamArgs& a, int64_t K, int swept,
                                 unsigned long long token, unsigned long long* mark, hipStream_t st) {
  const int n_chunks = (a.N + C - 1) / C;
  const int64_t n_wg = s.n_lists / (C == 32 ? WV / 8 : 1);
  const int64_t n_ids = sweep_grid(n_wg, n_chunks, swept);
  const int64_t long_waves = (int64_t)s.n_long * ((a.N + 63) / 64);
  const int64_t total = n_ids + (long_waves + WV - 1) / WV;
  if (long_waves > INT32_MAX || total > INT32_MAX) return hipErrorInvalidConfiguration;
  const uint64_t bytes = ((uint64_t)(K - 1) * (uint64_t)a.ldb + (uint64_t)a.N) * 4u;
  const PhaseStream ps{s.entries, s.uoff, s.pend, s.dest, s.n_lists / 2, s.phases, s.rows,
                       {s.entries, nullptr, nullptr, nullptr, nullptr, 0, s.lstart, s.lnblk, s.ldest, s.n_long}};
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL((spmm_phasesweep<C, WV>), dim3((unsigned)total), dim3(64 * WV), 0, st, ps, a.B, (uint32_t)bytes,
                     a.C, a.partial, a.N, (uint32_t)(a.ldb * 4), a.ldc, n_chunks, swept, a.relu, token, mark,
                     (int)n_ids);
  return hipGetLastError();
}

// Columns, waves per workgroup and mapping, from all of them on 26 matrices
// and widths (us; 32 columns put twice the rows in flight of 64, but a slice
// of B rows 1 or 2 KB apart uses few of an L2's channels; two workgroups of 8
// waves on a CU overlap one's phase start, where the misses are, with the
// other's, but keep two phases of B in the L2):
//   64 columns, pinned     few rows: uniform, 100000 of 30, N = 256: 221, 32
//                          columns of 8 / 16 waves 237 / 246; 30000 of 20: 62,
//                          73 / 73
//   32, 8 waves, swept     graphs with hubs (rows past the lists' average) and
//                          20 values a row: power-law, 116483 nodes, N = 256:
//                          245, 261 of 16 waves, 263 at 64; 58241: 190, 216,
//                          209; 232965: 988, 1055, 1005
//   32, 16 waves, swept    many rows, fewer values: 524288 nodes of 16, N = 256:
//                          1124, 8 waves 1188, 64 columns 1174; uniform, 300000
//                          of 8, N = 128: 119, 133, 135
//   32, 16 waves, pinned   where the memory-side cache does not hold a slice and
//                          the stream, which every chunk reads again (2^20
//                          nodes, N = 512, 134 + 340 MB: 8680, swept 9760)
static hipError_t launch_phasesweep(const ColSweep& s, const StreamArgs& a, int64_t K, unsigned long long token,
                                    unsigned long long* mark, hipStream_t st) {
  const int64_t rows = (int64_t)s.n_lists * s.rows;
  const bool cached = K * 128 + s.n_entries * 8 <= kMemCacheBytes;
  const bool hubs = s.n_long > 0 && s.n_entries >= 20 * rows;
  if (a.N % 32 || a.ldb % 32 || (rows < kSweptRows && !(cached && hubs)))
    return launch_phase_t<64, 16>(s, a, K, 0, token, mark, st);
  if (cached && hubs) return launch_phase_t<32, 8>(s, a, K, 1, token, mark, st);
  return launch_phase_t<32, 16>(s, a, K, cached, token, mark, st);
}

hipError_t launch_colsweep(const ColSweep& s, const StreamArgs& a, int64_t K, unsigned long long token,
                           unsigned long long* mark, hipStream_t st) {
  if (s.rows) return launch_phasesweep(s, a, K, token, mark, st);
  int cols, wv, swept;
  pick_launch((int64_t)s.n_lists * s.RL, s.RL, a, K, cols, wv, swept);
#define SRBCRS_SWEEP(C, RL, WV) return launch_t<C, RL, WV>(s, a, K, swept, token, mark, st)
#define SRBCRS_SWEEP_RL(C)                  \
  switch (s.RL) {                           \
    case 8:                                 \
      if (wv == 16) SRBCRS_SWEEP(C, 8, 16); \
      SRBCRS_SWEEP(C, 8, 1);                \
    case 4: SRBCRS_SWEEP(C, 4, 1);          \
    case 2: SRBCRS_SWEEP(C, 2, 1);          \
    default: SRBCRS_SWEEP(C, 1, 1);         \
  }
  if (cols == 32) SRBCRS_SWEEP_RL(32)
  SRBCRS_SWEEP_RL(64)
#undef SRBCRS_SWEEP_RL
#undef SRBCRS_SWEEP
}

static SweepTasks sweep_tasks(const ColSweepTasks& t) { return SweepTasks{t.begin, t.end, t.window, t.slot, t.n}; }

hipError_t launch_colsweep_repair(const ColSweepTasks& t, const StreamArgs& a, unsigned long long token,
                                  unsigned long long* mark, hipStream_t st) {
  const int64_t work = (int64_t)t.n * ((a.N + 63) / 64);
  if (work == 0) return hipSuccess;
  // every finite run launches them only to leave: 2048 waves cost 0.4 us less
  // than 4096, and a repair 13 % more (1024: 50 %)
  const unsigned grid = work < 2048 ? (unsigned)work : 2048u;
  hipLaunchKernelGGL(k_sweep_repair, dim3(grid), dim3(64), 0, st, mark, token, sweep_tasks(t), a.a_words, a.sidx,
                     a.a_packed, a.B, a.C, a.partial, a.rowmap, a.M, a.N, a.ldb, a.ldc, a.relu);
  return hipGetLastError();
}

static hipError_t build_phasesweep(const ColSweepIn& in, ColSweep& out, DeviceAlloc alloc, DeviceFree dfree,
                                   void* ctx, hipStream_t st) {
  const SweepTasks t = sweep_tasks(in.tasks);
  const int64_t rows = (int64_t)t.n * 16;
  const int64_t halves = (rows + 2 * out.rows - 1) / (2 * out.rows) * 2, slots = halves * out.rows;
  const int64_t per_list = in.n_values / (halves * 64);
  const int64_t long_len = std::max<int64_t>(128, per_list);   // as for the lists above
  if (rows == 0 || slots > INT32_MAX || long_len > 30000) return hipErrorInvalidValue;
  const int long_bin = sweep_bin((int)long_len);
  const int64_t long_cap = (in.n_values + in.n_values / 16 + 4096) / 128 + 1;
  out.phases = (int)std::min<int64_t>(kPhaseMax, std::max<int64_t>(1, per_list / kPhaseLoad));
  const int cap = (int)std::max<int64_t>(kPhaseLoad, (long_len + out.phases - 1) / out.phases);
  out.n_lists = (int)halves;
  int bin_shift = 0;
  while ((in.max_col >> bin_shift) >= kPhaseBins) ++bin_shift;
  const int64_t hp = halves * out.phases;
  std::vector<void*> temps;
  hipError_t err = hipSuccess;
  auto temp = [&](size_t bytes) {
    void* p = err == hipSuccess ? alloc(ctx, bytes) : nullptr;
    if (p)
      temps.push_back(p);
    else
      err = hipErrorOutOfMemory;
    return p;
  };
  out.bytes = 0;
  auto keep = [&](size_t n) {
    void* p = err == hipSuccess ? alloc(ctx, n) : nullptr;
    if (!p) err = hipErrorOutOfMemory;
    out.bytes += n;
    return p;
  };
  auto cleanup = [&](hipError_t e) {
    const bool idle = e == hipSuccess || hipStreamSynchronize(st) == hipSuccess;   // queued kernels may use these
    for (void* p : temps) dfree(ctx, p, idle);
    if (e != hipSuccess) {
      auto drop = [&](auto*& p) {
        if (p) dfree(ctx, (void*)p, idle);
        p = nullptr;
      };
      drop(out.entries);
      for (int** p : {&out.dest, &out.uoff, &out.pend, &out.lstart, &out.lnblk, &out.ldest}) drop(*p);
    }
    return e;
  };
  int* len = (int*)temp((size_t)rows * 4);
  int* hist = (int*)temp(2 * kSweepBins * 4);
  int* col_hist = (int*)temp(kPhaseBins * 4);
  uint8_t* phase_of = (uint8_t*)temp(kPhaseBins);
  int* vrow = (int*)temp((size_t)slots * 4);
  int* half_len = (int*)temp((size_t)halves * 4);
  int* lvrow = (int*)temp((size_t)long_cap * 4);
  // all entries, long rows, entries of the halves, values of the halves
  unsigned long long* total = (unsigned long long*)temp(32);
  uint16_t* cnt = (uint16_t*)temp((size_t)(slots * out.phases) * 2);
  uint32_t* place = (uint32_t*)temp((size_t)(slots * out.phases) * 4);
  uint16_t* load = (uint16_t*)temp((size_t)hp * 64 * 2);
  int* batches = (int*)temp((size_t)hp * 4);
  out.dest = (int*)keep((size_t)slots * 4);
  out.uoff = (int*)keep((size_t)(halves / 2 + 1) * 4);
  out.pend = (int*)keep((size_t)(halves / 2 * out.phases) * 4);
  out.lstart = (int*)keep((size_t)long_cap * 4);
  out.lnblk = (int*)keep((size_t)long_cap * 4);
  out.ldest = (int*)keep((size_t)long_cap * 4);
  if (err != hipSuccess) return cleanup(err);
#define SRBCRS_STEP(x)                          \
  do {                                          \
    const hipError_t e_ = (x);                  \
    if (e_ != hipSuccess) return cleanup(e_);   \
  } while (0)
  SRBCRS_STEP(hipMemsetAsync(hist, 0, 2 * kSweepBins * 4, st));
  SRBCRS_STEP(hipMemsetAsync(col_hist, 0, kPhaseBins * 4, st));
  SRBCRS_STEP(hipMemsetAsync(vrow, 0xff, (size_t)slots * 4, st));
  SRBCRS_STEP(hipMemsetAsync(out.dest, 0xff, (size_t)slots * 4, st));
  SRBCRS_STEP(hipMemsetAsync(half_len, 0, (size_t)halves * 4, st));
  SRBCRS_STEP(hipMemsetAsync(total, 0, 32, st));
  int64_t g = (rows + 31) / 32;
  hipLaunchKernelGGL(k_sweep_len, dim3((unsigned)(g > 8192 ? 8192 : g)), dim3(256), 0, st, t, in.words, in.sidx, len,
                     hist);
  SRBCRS_STEP(hipGetLastError());
  g = (rows + 256 * kSweepRankRows - 1) / (256 * kSweepRankRows);
  int* n_long = reinterpret_cast<int*>(total + 1);
  hipLaunchKernelGGL(k_sweep_rank, dim3((unsigned)g), dim3(256), 0, st, t, len, hist, hist + kSweepBins, (int)halves,
                     out.rows, long_bin, in.rowmap, in.M, vrow, out.dest, half_len, lvrow, out.ldest, (int)long_cap,
                     n_long);
  SRBCRS_STEP(hipGetLastError());
  g = (in.n_blocks + 256 * 16 - 1) / (256 * 16);
  hipLaunchKernelGGL(k_phase_hist, dim3((unsigned)(g > 1024 ? 1024 : g < 1 ? 1 : g)), dim3(256), 0, st, in.words,
                     in.sidx, in.n_blocks, bin_shift, col_hist);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_phase_cuts, dim3(1), dim3(1024), 0, st, col_hist, out.phases, phase_of);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_phase_count, dim3((unsigned)(slots / 8)), dim3(64), 0, st, t, in.words, in.sidx, vrow, out.rows,
                     out.phases, bin_shift, cap, phase_of, cnt);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_phase_assign, dim3((unsigned)hp), dim3(64), 0, st, cnt, out.rows, place, load, batches);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_phase_offsets, dim3(1), dim3(1024), 0, st, batches, half_len, (int)(halves / 2), out.phases,
                     out.pend, out.uoff, total);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_sweep_place_long, dim3((unsigned)((long_cap + 63) / 64)), dim3(64), 0, st, len, lvrow, n_long,
                     (int)long_cap, (int64_t)INT32_MAX, out.lstart, out.lnblk, total);
  SRBCRS_STEP(hipGetLastError());
  unsigned long long h[4] = {0, 0, 0, 0};
  SRBCRS_STEP(hipMemcpyAsync(h, total, 32, hipMemcpyDeviceToHost, st));
  SRBCRS_STEP(hipStreamSynchronize(st));
  out.n_long = (int)(h[1] & 0xffffffffu);
  out.n_entries = (int64_t)h[0];
  if (h[0] > (unsigned long long)INT32_MAX - 64 || out.n_long > long_cap || h[2] > h[3] + h[3] / 2 + 65536)
    return cleanup(hipErrorInvalidValue);
  out.entries = (uint2*)keep(((size_t)h[0] + 8) * 8);
  if (!out.entries) return cleanup(hipErrorOutOfMemory);
  const PhaseFill f{cnt, place, load, out.uoff, out.pend, out.rows, out.phases};
  hipLaunchKernelGGL(k_phase_fill, dim3((unsigned)(slots / 8)), dim3(64), 0, st, t, in.words, in.sidx, in.packed, vrow,
                     f, out.entries);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_phase_pad, dim3((unsigned)(halves / 2 * out.phases)), dim3(128), 0, st, f, out.entries);
  SRBCRS_STEP(hipGetLastError());
  if (out.n_long) {
    hipLaunchKernelGGL(k_sweep_fill, dim3((unsigned)((out.n_long + 7) / 8)), dim3(64), 32 * 4, st, t, in.words,
                       in.sidx, in.packed, vrow, (int64_t)0, 1, half_len, out.uoff, out.uoff, 1, 31, lvrow, len,
                       out.lstart, out.lnblk, n_long, (int)long_cap, out.entries);
    SRBCRS_STEP(hipGetLastError());
  }
  SRBCRS_STEP(hipStreamSynchronize(st));
#undef SRBCRS_STEP
  return cleanup(hipSuccess);
}

hipError_t build_colsweep(const ColSweepIn& in, ColSweep& out, DeviceAlloc alloc, DeviceFree dfree, void* ctx,
                          hipStream_t st) {
  if (out.rows) return build_phasesweep(in, out, alloc, dfree, ctx, st);
  const SweepTasks t = sweep_tasks(in.tasks);
  const int64_t rows = (int64_t)t.n * 16;
  const int RL = out.RL;
  const int64_t n_lists = (rows + 8 * RL - 1) / (8 * RL) * 8, slots = n_lists * RL;
  if (rows == 0 || slots > INT32_MAX) return hipErrorInvalidValue;
  out.n_lists = (int)n_lists;
  // rows over the lists' average, and over 128 values, are long (power-law
  // graph of 8000 nodes, N = 64, us: 88 none, 28 over 256, 21 over 128; of
  // 232965 nodes, N = 256: 1378 over twice the average, 1297 over it)
  constexpr int64_t kLongMin = 128;
  const int64_t long_len = std::max<int64_t>(kLongMin, in.n_values / n_lists);
  const int long_bin = sweep_bin((int)long_len);
  // stored values, and room for explicit zeros (k_sweep_len counts them)
  const int64_t most = in.n_values + in.n_values / 16 + 4096;
  const int64_t long_cap = most / kLongMin + 1;   // rows past kLongMin values
  // Small streams take room for the most their lists may need, which saves a
  // wait for the sum (25 us of the 110 of a 4096-row matrix); large ones, where
  // it would be a third more than they need, wait.
  int64_t cap = most + kSweepBatch * n_lists + kSweepLongBatch * long_cap;
  const bool ahead = cap * 8 <= (16 << 20);
  if (!ahead) cap = INT32_MAX;
  int *len = nullptr, *hist = nullptr, *vrow = nullptr, *list_len = nullptr, *lvrow = nullptr;
  unsigned long long* total = nullptr;
  bool idle = true;
  auto drop = [&](auto*& p) {
    if (p) dfree(ctx, (void*)p, idle);
    p = nullptr;
  };
  auto cleanup = [&](hipError_t e) {
    idle = e == hipSuccess || hipStreamSynchronize(st) == hipSuccess;   // queued kernels may use these
    drop(len);
    drop(hist);
    drop(vrow);
    drop(list_len);
    drop(lvrow);
    drop(total);
    if (e != hipSuccess) {
      drop(out.entries);
      for (int** p : {&out.start, &out.nblk, &out.wblk8, &out.wblk4, &out.dest, &out.lstart, &out.lnblk, &out.ldest})
        drop(*p);
    }
    return e;
  };
  bool room = true;
  auto temp = [&](size_t bytes) {
    void* p = room ? alloc(ctx, bytes) : nullptr;
    room = p != nullptr;
    return p;
  };
  out.bytes = 0;
  auto keep = [&](size_t bytes) {
    out.bytes += bytes;
    return temp(bytes);
  };
  len = (int*)temp((size_t)rows * 4);
  hist = (int*)temp(2 * kSweepBins * 4);
  vrow = (int*)temp((size_t)slots * 4);
  list_len = (int*)temp((size_t)n_lists * 4);
  lvrow = (int*)temp((size_t)long_cap * 4);
  total = (unsigned long long*)temp(16);   // entries taken, long rows
  out.start = (int*)keep((size_t)n_lists * 4);
  out.nblk = (int*)keep((size_t)n_lists * 4);
  out.wblk8 = (int*)keep((size_t)n_lists / 8 * 4);
  out.wblk4 = (int*)keep((size_t)n_lists / 4 * 4);
  out.dest = (int*)keep((size_t)slots * 4);
  out.lstart = (int*)keep((size_t)long_cap * 4);
  out.lnblk = (int*)keep((size_t)long_cap * 4);
  out.ldest = (int*)keep((size_t)long_cap * 4);
  if (ahead) out.entries = (uint2*)keep((size_t)(cap + 8) * 8);
  if (!room) return cleanup(hipErrorOutOfMemory);
#define SRBCRS_STEP(x)                          \
  do {                                          \
    const hipError_t e_ = (x);                  \
    if (e_ != hipSuccess) return cleanup(e_);   \
  } while (0)
  SRBCRS_STEP(hipMemsetAsync(hist, 0, 2 * kSweepBins * 4, st));
  SRBCRS_STEP(hipMemsetAsync(vrow, 0xff, (size_t)slots * 4, st));
  SRBCRS_STEP(hipMemsetAsync(out.dest, 0xff, (size_t)slots * 4, st));
  SRBCRS_STEP(hipMemsetAsync(list_len, 0, (size_t)n_lists * 4, st));
  SRBCRS_STEP(hipMemsetAsync(total, 0, 16, st));
  int64_t g = (rows + 31) / 32;
  hipLaunchKernelGGL(k_sweep_len, dim3((unsigned)(g > 8192 ? 8192 : g)), dim3(256), 0, st, t, in.words, in.sidx, len,
                     hist);
  SRBCRS_STEP(hipGetLastError());
  g = (rows + 256 * kSweepRankRows - 1) / (256 * kSweepRankRows);
  int* n_long = reinterpret_cast<int*>(total + 1);
  hipLaunchKernelGGL(k_sweep_rank, dim3((unsigned)g), dim3(256), 0, st, t, len, hist, hist + kSweepBins, (int)n_lists,
                     RL, long_bin, in.rowmap, in.M, vrow, out.dest, list_len, lvrow, out.ldest, (int)long_cap, n_long);
  SRBCRS_STEP(hipGetLastError());
  const int n8 = (int)(n_lists / 8);
  hipLaunchKernelGGL(k_sweep_place, dim3((unsigned)((n8 + 63) / 64)), dim3(64), 0, st, list_len, n8, cap, out.start,
                     out.nblk, out.wblk8, out.wblk4, total);
  SRBCRS_STEP(hipGetLastError());
  hipLaunchKernelGGL(k_sweep_place_long, dim3((unsigned)((long_cap + 63) / 64)), dim3(64), 0, st, len, lvrow, n_long,
                     (int)long_cap, cap, out.lstart, out.lnblk, total);
  SRBCRS_STEP(hipGetLastError());
  unsigned long long h_total[2] = {0, 0};
  auto fetch_total = [&]() -> hipError_t {
    const hipError_t e = hipMemcpyAsync(h_total, total, 16, hipMemcpyDeviceToHost, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
  };
  auto fits = [&] {
    out.n_long = (int)(h_total[1] & 0xffffffffu);
    out.n_entries = (int64_t)h_total[0];
    return h_total[0] <= (unsigned long long)cap - (ahead ? 0 : 64) && out.n_long <= long_cap;
  };
  if (!ahead) {
    SRBCRS_STEP(fetch_total());
    if (!fits()) return cleanup(hipErrorInvalidValue);
    out.entries = (uint2*)keep((size_t)(out.n_entries + 8) * 8);
    if (!room) return cleanup(hipErrorOutOfMemory);
  }
  const int64_t longs = ahead ? long_cap : out.n_long;
  hipLaunchKernelGGL(k_sweep_fill, dim3((unsigned)((slots + 7) / 8 + (longs + 7) / 8)), dim3(64),
                     32 * out.phases * 4, st, t, in.words, in.sidx, in.packed, vrow, slots, RL, list_len, out.start,
                     out.nblk, out.phases, out.shift, lvrow, len, out.lstart, out.lnblk, n_long, (int)long_cap,
                     out.entries);
  SRBCRS_STEP(hipGetLastError());
  SRBCRS_STEP(ahead ? fetch_total() : hipStreamSynchronize(st));
#undef SRBCRS_STEP
  return cleanup(fits() ? hipSuccess : hipErrorInvalidValue);
}

}  // namespace srbcrs
