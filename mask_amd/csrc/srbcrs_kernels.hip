// Host launchers of the SR-BCRS kernels (templates in srbcrs_stream.hpp).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "srbcrs_kernels.h"
#include "srbcrs_stream.hpp"  // segment_reduce, zero_rows, csr_spmm_rowwave

namespace srbcrs {

// ---------------------------------------------------------------------------
// Host launchers.

hipError_t launch_row(const StreamArgs& a, const int* soff, int Mo, int vec, const RunOpts& o,
                      hipStream_t st) {
  return (o.a_compact && a.a_words) ? launch_row_compact(a, soff, Mo, vec, o, st)
                                    : launch_row_dense(a, soff, Mo, vec, o, st);
}

hipError_t launch_tasks(const StreamArgs& a, const TaskTable& t, int vec, const RunOpts& o,
                        hipStream_t st) {
  return (o.a_compact && a.a_words) ? launch_tasks_compact(a, t, vec, o, st)
                                    : launch_tasks_dense(a, t, vec, o, st);
}

hipError_t launch_reduce(const ReduceArgs& a, int vec, hipStream_t st) {
  if (a.n_red == 0) return hipSuccess;
  const int64_t total = (int64_t)a.n_red * a.tile_rows * (a.N / vec);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (vec == 4)
    hipLaunchKernelGGL(segment_reduce<4>, dim3((unsigned)blocks), dim3(256), 0, st, a.partial, a.C,
                       a.red_window, a.red_slot_off, a.n_red, a.tile_rows, a.M, a.N, a.ldc, a.rowmap, a.relu);
  else if (vec == 2)
    hipLaunchKernelGGL(segment_reduce<2>, dim3((unsigned)blocks), dim3(256), 0, st, a.partial, a.C,
                       a.red_window, a.red_slot_off, a.n_red, a.tile_rows, a.M, a.N, a.ldc, a.rowmap, a.relu);
  else
    hipLaunchKernelGGL(segment_reduce<1>, dim3((unsigned)blocks), dim3(256), 0, st, a.partial, a.C,
                       a.red_window, a.red_slot_off, a.n_red, a.tile_rows, a.M, a.N, a.ldc, a.rowmap, a.relu);
  return hipGetLastError();
}

template <int C>
static hipError_t launch_csr_t(const CsrArgs& a, uint32_t bytes, hipStream_t st) {
  const int n_chunks = (a.N + C - 1) / C;
  const int64_t n_wg = ((int64_t)a.M + 1024 / C - 1) / (1024 / C);
  int64_t grid = n_wg * n_chunks;
  if (n_chunks <= kNumXcd && kNumXcd % n_chunks == 0) {
    const int per = kNumXcd / n_chunks;
    grid = (n_wg + per - 1) / per * kNumXcd;
  }
  if (grid > INT32_MAX) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((csr_spmm_rowgroup<C>), dim3((unsigned)grid), dim3(256), 0, st, a.rowptr, a.colind, a.values, a.B,
                     bytes, a.C, a.M, a.N, (uint32_t)(a.ldb * 4), a.ldc, n_chunks, (int)n_wg);
  return hipGetLastError();
}

// vec: columns per lane per pass of the wave kernel (64*vec divides N, or 1).
hipError_t launch_csr(const CsrArgs& a, int vec, hipStream_t st) {
  if (a.M == 0) return hipSuccess;
  const uint64_t bytes = a.K > 0 ? ((uint64_t)(a.K - 1) * (uint64_t)a.ldb + (uint64_t)a.N) * 4u : 0u;
  const bool quads = a.N % 4 == 0 && a.ldb % 4 == 0 && a.ldc % 4 == 0 && reinterpret_cast<uintptr_t>(a.B) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(a.C) % 16 == 0;
  // One row per lane group wherever float4 segments and 32-bit offsets fit,
  // but on B so tall that no cache holds any of it, where whole 1 KB segments
  // of a row per wave gather a little faster (100000 x 400000, 12 per row, N =
  // 256: 186 / 195 us; at 384 columns, not whole segments, 355 / 280).  32
  // columns where their slice of B is within reach of the L2 (K = 65536: 138 us,
  // 64 columns 153; 150000: 184 / 176), 64 where theirs is in it (K = 8000: 18,
  // 32 columns 20) or 32-column segments straddle cache lines (N = 100: 98 / 125).
  if (quads && !(vec == 4 && a.K > 262144) && a.K < (int64_t(1) << 32) &&
      bytes + (uint64_t)a.N * 4 < (uint64_t(1) << 32)) {
    if (a.N % 32 || a.ldb % 32 || a.K <= 16384 || a.K > 131072) return launch_csr_t<64>(a, (uint32_t)bytes, st);
    return launch_csr_t<32>(a, (uint32_t)bytes, st);
  }
  const int n_chunks = (a.N + 64 * vec - 1) / (64 * vec);
  const int64_t nwg = ((int64_t)a.M + 3) / 4 * n_chunks;
  if (nwg == 0) return hipSuccess;
  if (nwg > INT32_MAX) return hipErrorInvalidConfiguration;
  dim3 grid((unsigned)nwg);
  if (vec == 4)
    hipLaunchKernelGGL((csr_spmm_rowwave<4, 8>), grid, dim3(256), 0, st, a.rowptr, a.colind,
                       a.values, a.B, a.C, a.M, a.N, a.ldb, a.ldc, n_chunks);
  else if (vec == 2)
    hipLaunchKernelGGL((csr_spmm_rowwave<2, 8>), grid, dim3(256), 0, st, a.rowptr, a.colind,
                       a.values, a.B, a.C, a.M, a.N, a.ldb, a.ldc, n_chunks);
  else
    hipLaunchKernelGGL((csr_spmm_rowwave<1, 8>), grid, dim3(256), 0, st, a.rowptr, a.colind,
                       a.values, a.B, a.C, a.M, a.N, a.ldb, a.ldc, n_chunks);
  return hipGetLastError();
}

hipError_t launch_zero_rows(float* C, const int* rows, int n_rows, int N, int64_t ldc, hipStream_t st) {
  if (n_rows == 0 || N == 0) return hipSuccess;
  const int64_t total = (int64_t)n_rows * N;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(zero_rows<float>, dim3((unsigned)blocks), dim3(256), 0, st, C, rows, n_rows, N, ldc);
  return hipGetLastError();
}

}  // namespace srbcrs
