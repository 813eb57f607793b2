"""The column sweep (the default launch at low block fill, from a plan's
second run on): the block kernels' bits on every schedule, width and row
order, infinities and NaNs included, under graph capture and on two streams."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import assert_gate, gate, random_csr

pytestmark = pytest.mark.gpu

# (M, K, columns per row, heavy rows): lists shorter than a wave, one row past a window, several list
# heights, one and many column phases, rows long enough to leave the lists
SHAPES = [(1, 300, 200, 0), (17, 3000, 16, 0), (129, 5000, 20, 2), (1025, 20000, 14, 3), (5003, 40011, 13, 5)]
WIDTHS = [16, 48, 64, 112, 256]


def _csr(M, K, per_row, heavy, seed):
    rng = np.random.default_rng(seed)
    rows = [np.sort(rng.choice(K, min(K, 2000 if r < heavy else int(rng.integers(per_row // 2, 2 * per_row))),
                               replace=False)) for r in range(M)]
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    colind = np.concatenate(rows).astype(np.int32)
    return rowptr, colind, rng.uniform(-1, 1, colind.size).astype(np.float32)


def _plan(csr, M, **kw):
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    return Plan(*(torch.from_numpy(np.asarray(a)).cuda() for a in csr), M, **kw)


def _same(a, b):
    """Equal bits of value: NaN where NaN, else equal."""
    import torch
    na, nb = torch.isnan(a), torch.isnan(b)
    return torch.equal(na, nb) and torch.equal(a[~na], b[~nb])


def _check(plan, B, what, **kw):
    ref = plan.run(B, grid_order=1, depth=2, wg_cols=128, **kw)
    for i in range(3):   # the first run may take the block kernel, the later ones the sweep
        assert _same(plan.run(B, **kw), ref), (what, i)
    return ref


@pytest.mark.parametrize("policy", [("row", 0), ("auto", 0), ("split", 7), ("strict_lb", 9), ("multi_bind", 0)])
@pytest.mark.parametrize("shape", SHAPES)
def test_bits_of_the_block_kernels(gpu, shape, policy):
    import torch
    M, K, per_row, heavy = shape
    csr = _csr(M, K, per_row, heavy, M)
    plan = _plan(csr, M)
    plan.set_schedule(*policy)
    for N in WIDTHS:
        print("[case] colsweep", shape, policy, N, flush=True)
        B = torch.from_numpy(np.random.default_rng(N).uniform(-1, 1, (K, N)).astype(np.float32)).cuda()
        C = _check(plan, B, (shape, policy, N))
        _check(plan, B, (shape, policy, N, "relu"), relu=True)
    assert_gate(gate(C.cpu().numpy(), *csr, B.cpu().numpy(), M))


def test_second_run_builds_the_stream(gpu):
    """The stream (8 bytes per stored value) is allocated by the second run."""
    import torch
    M = K = 60000
    rng = np.random.default_rng(1)
    cols = np.sort(rng.integers(0, K // 16, (M, 16)) * 16 + np.arange(16), axis=1)
    csr = (np.arange(M + 1, dtype=np.int32) * 16, cols.ravel().astype(np.int32),
           rng.uniform(-1, 1, M * 16).astype(np.float32))
    plan = _plan(csr, M)
    B, out = torch.ones((K, 64), device="cuda"), torch.empty((M, 64), device="cuda")
    free = []
    plan.trim()   # gives back the device memory kept from the conversion, which the stream would take
    for _ in range(3):
        print("[case] stream build", flush=True)
        plan.run(B, out)
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - free[1] >= 8 * M * 16 and free[2] == free[1]


# (M, K, columns per row, N, band): 64 columns with a ragged last chunk; 32 columns with 16 waves, all XCDs
# on one chunk and chunks pinned; with 8 waves; rows whose columns all lie in one phase; mostly empty rows
@pytest.mark.parametrize("policy", [("row", 0), ("split", 5)])
@pytest.mark.parametrize("shape", [(6100, 50000, 9, 1008, 0), (210001, 49999, 4, 32, 0), (210000, 1990000, 4, 32, 0),
                                   (66001, 52000, 30, 128, 0), (70003, 70003, 20, 128, 200),
                                   (150000, 49160, 1, 128, 0)])
def test_phase_sweep(gpu, shape, policy):
    """Widths and sizes at which the workgroups' rows are pooled."""
    import torch
    M, K, per_row, N, band = shape
    rng = np.random.default_rng(M + per_row)
    lens = rng.integers(0, 2 * per_row + 1, M)
    lens[[5, M // 2]] = 3000    # longer than a list
    lens[17:40] = 130           # more than a phase's share
    row = np.repeat(np.arange(M), lens)
    cols = rng.integers(0, K, row.size) if not band else np.clip(row + rng.integers(-band, band, row.size), 0, K - 1)
    cols = cols[np.lexsort((cols, row))].astype(np.int32)
    csr = (np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), cols,
           rng.uniform(-1, 1, row.size).astype(np.float32))
    print("[case] phase sweep", shape, policy, row.size, flush=True)
    plan = _plan(csr, M)
    plan.set_schedule(*policy)
    B = torch.rand((K, N), device="cuda") - 0.5
    _check(plan, B, shape)
    _check(plan, B, (shape, "relu"), relu=True)
    B[int(cols[777]), 7] = float("inf")
    assert not bool(torch.isfinite(_check(plan, B, (shape, "inf"))).all())


# (M, K, columns per row, N): lists of 4 rows (too few rows for 8), and lists of 8 in workgroups of 16 waves in
# step (more columns than the phase sweep's entries can name) at 32 and at 64 columns
@pytest.mark.parametrize("shape", [(60000, 60000, 16, 64), (240500, 2_200_000, 8, 32), (120500, 2_200_000, 8, 48)])
def test_list_layouts(gpu, shape):
    """The list layouts and launches that the other shapes here do not take."""
    import torch
    M, K, per_row, N = shape
    rng = np.random.default_rng(M)
    lens = rng.integers(0, 2 * per_row + 1, M)
    lens[[7, M // 3]] = 2000    # rows outside the lists
    cols = rng.integers(0, K, int(lens.sum()))
    row = np.repeat(np.arange(M), lens)
    cols = cols[np.lexsort((cols, row))].astype(np.int32)
    csr = (np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), cols,
           rng.uniform(-1, 1, cols.size).astype(np.float32))
    print("[case] list layouts", shape, cols.size, flush=True)
    plan = _plan(csr, M)
    B = torch.rand((K, N), device="cuda") - 0.5
    _check(plan, B, shape)
    _check(plan, B, (shape, "relu"), relu=True)
    B[int(cols[777]), 7] = float("nan")
    assert not bool(torch.isfinite(_check(plan, B, (shape, "nan"))).all())


@pytest.mark.parametrize("K,N,built", [(300000, 256, False), (300000, 224, True), (60000, 256, True)])
def test_short_rows_without_shared_columns(gpu, K, N, built):
    """Ten values a row and under two a column at whole 64-column chunks: the
    block kernels stay, and no stream is built."""
    import torch
    M = 20000
    rng = np.random.default_rng(K)
    cols = np.sort(rng.integers(0, K, (M, 10)), axis=1).astype(np.int32).ravel()
    cols[-1] = K - 1
    plan = _plan((np.arange(M + 1, dtype=np.int32) * 10, cols, rng.uniform(-1, 1, M * 10).astype(np.float32)), M)
    print("[case] short rows", K, N, flush=True)
    B, out = torch.rand((K, N), device="cuda"), torch.empty((M, N), device="cuda")
    plan.trim()
    plan.run(B, out)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan.run(B, out)
    torch.cuda.synchronize()
    assert (torch.cuda.mem_get_info()[0] < free) == built
    _check(plan, B, (K, N))


@pytest.mark.parametrize("policy", [("row", 0), ("split", 7)])
def test_non_finite_dense_values(gpu, policy):
    """An infinity or NaN of B poisons every row of the windows whose blocks
    hold its column, as in the block kernels: also a column whose only entry
    is an explicit zero, and one past a list's end; a later finite run is not
    affected."""
    import torch
    M, K, N = 1025, 20000, 64
    rowptr, colind, values = _csr(M, K, 14, 2, 3)
    values[5:400:7] = 0.0                     # explicit zeros, dropped from the compact values
    zero_col = int(colind[5])
    plan = _plan((rowptr, colind, values), M)
    plan.set_schedule(*policy)
    fine = torch.from_numpy(np.random.default_rng(2).uniform(-1, 1, (K, N)).astype(np.float32)).cuda()
    for cols, v in (((int(colind[700]), zero_col), float("inf")), ((int(colind[-1]),), float("nan")),
                    ((zero_col,), float("-inf"))):
        B = fine.clone()
        B[list(cols), 3] = v
        B[list(cols), 63] = -v
        print("[case] non-finite", policy, cols, v, flush=True)
        ref = _check(plan, B, (cols, v))
        assert bool(torch.isnan(ref).any())
        _check(plan, B, (cols, v, "relu"), relu=True)
        _check(plan, fine, "finite again")


@pytest.mark.parametrize("policy", [("row", 0), ("split", 7)])
@pytest.mark.parametrize("N", [16, 48, 112, 256])
def test_non_finite_at_every_width(gpu, N, policy):
    """The repair pass over chunks that end inside 64 columns, a last window
    that is not whole, windows without a block, and a row order."""
    import torch
    M, K = 1501, 20000
    rowptr, colind, values = _csr(M, K, 14, 2, N)
    empty = np.repeat(np.arange(M) // 16 % 9 == 4, np.diff(rowptr))   # the windows 4, 13, ... hold nothing
    lens = np.where(np.arange(M) // 16 % 9 == 4, 0, np.diff(rowptr))
    csr = (np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), colind[~empty], values[~empty])
    B = torch.from_numpy(np.random.default_rng(N).uniform(-1, 1, (K, N)).astype(np.float32)).cuda()
    B[csr[1][::97].astype(np.int64), N // 2] = float("inf")
    B[csr[1][5:9].astype(np.int64), N - 1] = float("nan")
    for kw in ({}, dict(row_order="first_col_sort", K=K)):
        plan = _plan(csr, M, **kw)
        plan.set_schedule(*policy)
        print("[case] non-finite width", N, policy, kw, flush=True)
        assert not bool(torch.isfinite(_check(plan, B, (N, policy, kw))).all())
        _check(plan, B, (N, policy, kw, "relu"), relu=True)


@pytest.mark.parametrize("order", ["first_col_sort", "sparse_rows"])
def test_row_orders_and_strides(gpu, order):
    import torch
    M, K, N = 700, 9000, 96
    csr = random_csr(M, K, 0.002, seed=5, empty_rows=0.2, heavy_rows=2, heavy_len=900)
    plan = _plan(csr, M, row_order=order, K=K)
    wide = torch.from_numpy(np.random.default_rng(5).uniform(-1, 1, (K, 131)).astype(np.float32)).cuda()
    for ldb, ldc in ((96, 96), (100, 104), (131, 96), (96, 101)):   # the last two: the block kernels
        B = torch.as_strided(wide.flatten()[: K * ldb].clone(), (K, N), (ldb, 1))
        print("[case] order", order, ldb, ldc, flush=True)
        ref = plan.run(B, grid_order=1, depth=2, wg_cols=128)
        for _ in range(3):
            C = torch.full((M, ldc), 7.0, device="cuda")
            plan.run(B, C[:, :N])
            assert torch.equal(C[:, :N], ref) and bool((C[:, N:] == 7.0).all())


def test_capture_and_two_streams(gpu):
    """Captured before and after the stream is built, replays equal the eager
    results; two streams share one plan, one of them with NaNs."""
    import torch
    M, K, N = 3000, 30000, 128
    csr = _csr(M, K, 15, 3, 9)
    rng = np.random.default_rng(9)
    mk = lambda: torch.from_numpy(rng.uniform(-1, 1, (K, N)).astype(np.float32)).cuda()
    for eager in (1, 2):
        plan = _plan(csr, M)
        B, C = mk(), torch.empty((M, N), device="cuda")
        for _ in range(eager):
            plan.run(B, C)
        torch.cuda.synchronize()
        print("[case] capture after", eager, flush=True)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            plan.run(B, C)
        for i in range(4):
            B.copy_(mk())
            if i == 2:
                B[int(csr[1][40])] = float("nan")
            C.fill_(7.0)
            g.replay()
            torch.cuda.synchronize()
            assert _same(C, plan.run(B, grid_order=1, depth=2, wg_cols=128)), (eager, i)
    B1, B2 = mk(), mk()
    B2[int(csr[1][40])] = float("nan")
    r1, r2 = (plan.run(b, grid_order=1, depth=2, wg_cols=128) for b in (B1, B2))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    print("[case] two streams", flush=True)
    outs = []
    for _ in range(20):
        for s, b in ((s1, B1), (s2, B2)):
            with torch.cuda.stream(s):
                outs.append(plan.run(b))
    torch.cuda.synchronize()
    assert all(_same(o, (r1, r2)[i % 2]) for i, o in enumerate(outs))


@pytest.mark.parametrize("M,per_row,N", [(65536, 16, 512), (20000, 20, 128)])   # a phase stream, a list stream
def test_replay_after_a_non_finite_one(gpu, M, per_row, N):
    """A captured run repairs the replays whose own sums are not finite and no
    others: the ones after take as long as before."""
    import torch
    rng = np.random.default_rng(M)
    cols = np.sort(rng.integers(0, M, (M, per_row)), axis=1).astype(np.int32).ravel()
    plan = _plan((np.arange(M + 1, dtype=np.int32) * per_row, cols, rng.uniform(-1, 1, cols.size).astype(np.float32)), M)
    fine = torch.rand((M, N), device="cuda") - 0.5
    bad = fine.clone()
    bad[int(cols[7])] = float("inf")
    B, C = fine.clone(), torch.empty((M, N), device="cuda")
    for _ in range(2):
        plan.run(B, C)
    refs = [plan.run(b, grid_order=1, depth=2, wg_cols=128) for b in (fine, bad)]
    torch.cuda.synchronize()
    print("[case] replays", M, per_row, N, flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.run(B, C)

    def replay(i):
        B.copy_((fine, bad)[i])
        C.fill_(7.0)
        g.replay()
        assert _same(C, refs[i])
        best = float("inf")
        for _ in range(10):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            g.replay()
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]))
        plan.run(B)   # eager work between replays
        return best

    before = replay(0)
    for _ in range(2):
        replay(1)
        # (a repair pass more than doubles a replay)
        assert replay(0) < 1.5 * before + 0.01


def test_widths_that_share_streams(gpu):
    """Once a schedule's streams hold as much as the block values, a width runs
    on the stream of another one, of either kind: the same bits."""
    import torch
    M = K = 65536
    rng = np.random.default_rng(11)
    cols = np.sort(rng.integers(0, K, (M, 16)), axis=1).astype(np.int32).ravel()
    plan = _plan((np.arange(M + 1, dtype=np.int32) * 16, cols, rng.uniform(-1, 1, cols.size).astype(np.float32)), M)
    wide = torch.rand((K, 512), device="cuda") - 0.5
    plan.trim()
    torch.cuda.synchronize()
    out, free = torch.empty((M, 512), device="cuda"), torch.cuda.mem_get_info()[0]
    widths = list(range(512, 95, -32)) + [80, 64, 48, 32, 16]
    for N in widths:
        for _ in range(2):
            plan.run(wide[:, :N], out[:, :N])
    plan.trim()   # the builds' temporaries
    streams = free - torch.cuda.mem_get_info()[0]
    assert 2 * 8 * cols.size < streams < plan.total_blocks * 512 + 8 * cols.size, streams
    for N in widths:
        print("[case] shared stream", N, flush=True)
        _check(plan, wide[:, :N].contiguous(), N)


def test_more_captured_runs_than_marks(gpu):
    """Runs recorded past the 1024th of a plan have no mark of their own: their
    replays are repaired as well."""
    import torch
    M = K = 2000
    csr = _csr(M, K, 20, 2, 4)
    plan = _plan(csr, M)
    fine = torch.rand((K, 64), device="cuda") - 0.5
    bad = fine.clone()
    bad[int(csr[1][7])] = float("inf")
    B, C = fine.clone(), [torch.empty((M, 64), device="cuda") for _ in range(2)]
    refs = [plan.run(b, grid_order=1, depth=2, wg_cols=128) for b in (fine, bad)]
    for _ in range(2):
        plan.run(B, C[0])
    torch.cuda.synchronize()
    print("[case] more captured runs than marks", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(1030):
            plan.run(B, C[0])
        plan.run(B, C[1])
    for i in (0, 1, 0, 1, 0):
        B.copy_((fine, bad)[i])
        for c in C:
            c.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        assert all(_same(c, refs[i]) for c in C), i
        plan.run(B)   # eager work between replays
