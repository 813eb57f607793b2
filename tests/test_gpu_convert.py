"""Device-side conversion (is_device = 1) against the oracle, bit for bit,
and against the host conversion of the same device CSR (is_device = 2)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle
from tests.helpers import random_csr

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


def _arrays(plan):
    import torch
    from mask_amd import _capi
    n = plan.row_windows + 1
    soff = torch.empty(n, dtype=torch.int32, device="cuda")
    sidx = torch.empty(max(plan.total_blocks * plan.blk_w, 1), dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    _capi.check(_capi.lib().srbcrs_plan_export_index(plan.handle, soff.data_ptr(), n, sidx.data_ptr(),
                                                     sidx.numel(), st))
    bp = torch.zeros(max(plan.row_windows, 1), dtype=torch.int32, device="cuda")
    e2c = torch.zeros(max(plan.nnz, 1), dtype=torch.int32, device="cuda")
    e2r = torch.zeros(max(plan.nnz, 1), dtype=torch.int32, device="cuda")
    _capi.check(_capi.lib().srbcrs_plan_write_edges(plan.handle, bp.data_ptr(), plan.row_windows, e2c.data_ptr(),
                                                    plan.nnz, e2r.data_ptr(), plan.nnz, st))
    val = plan.block_values()
    torch.cuda.synchronize()
    return dict(soff=soff.cpu().numpy(), sidx=sidx.cpu().numpy()[: plan.total_blocks * plan.blk_w],
                val=val.cpu().numpy(), block_partition=bp.cpu().numpy()[: plan.row_windows],
                edge_to_col=e2c.cpu().numpy()[: plan.nnz], edge_to_row=e2r.cpu().numpy()[: plan.nnz],
                total=plan.total_blocks, max_col=plan.max_col)


def _same(a, b):
    assert a["total"] == b["total"]
    for k in ("soff", "sidx", "block_partition", "edge_to_row", "edge_to_col"):
        assert np.array_equal(a[k], b[k]), k
    assert a["val"].tobytes() == b["val"].tobytes()


def _cases():
    yield "tiny", random_csr(1, 1, 1.0, 0)
    yield "m17", random_csr(17, 40, 0.2, 1)
    yield "unsorted-dup", random_csr(203, 700, 0.03, 2, unsorted=True, duplicates=True, empty_rows=0.2)
    yield "skewed", random_csr(500, 3000, 0.01, 3, heavy_rows=5, heavy_len=2500, empty_rows=0.3)
    yield "empty", (np.zeros(33, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32))


@pytest.mark.parametrize("blk", [(16, 8), (32, 32)])
def test_device_conversion_matches_oracle(gpu, blk):
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    for name, (rp, ci, vv) in _cases():
        M = rp.shape[0] - 1
        _say("convert", name, blk, M, ci.size)
        t = lambda a: torch.from_numpy(a).cuda()
        dev = _arrays(Plan(t(rp), t(ci), t(vv), M, blk[0], blk[1], convert_on="device"))
        host = _arrays(Plan(t(rp), t(ci), t(vv), M, blk[0], blk[1], convert_on="host"))
        o = oracle.convert(rp, ci, vv, M, blk[0], blk[1])
        _same(dev, o)
        _same(host, o)
        assert dev["max_col"] == (int(ci.max()) if ci.size else -1)


@pytest.mark.parametrize("name", ["uniform-65536", "banded-524288", "rmat-2^20", "gcn-232965"])
def test_device_conversion_workloads(gpu, name):
    import torch
    from mask_amd import datasets
    from mask_amd.SRBCRSSpMM import Plan
    m = datasets.make_config(name, scale_down=8)
    _say("convert workload", name, m.M, m.nnz)
    t = lambda a: torch.from_numpy(a).cuda()
    _same(_arrays(Plan(t(m.rowptr), t(m.colind), t(m.values), m.M)), oracle.convert(m.rowptr, m.colind, m.values, m.M))


@pytest.mark.parametrize("blk,K", [((16, 8), 300), ((16, 8), 3_000_000), ((32, 32), 70_000)])
def test_device_conversion_window_lengths(gpu, blk, K):
    """Windows at the edges of the converter's length classes, several past the last one."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    rng = np.random.default_rng(K)
    lens = [0, 1, 63, 257, 2047, 2048, 2049, 4095, 4096, 4097, 16383, 16384, 16385, 20000, 0, 50000, 16390]
    lens += [0] * 300 + [9]
    M = len(lens) * blk[0] - 5
    counts = []
    for w, n in enumerate(lens):   # edges over the window's rows: some empty, duplicates and unsorted columns
        rows = min(blk[0], M - w * blk[0])
        counts.append(np.bincount(rng.integers(0, rows, n) // 2 * 2 % rows, minlength=rows))
    rp = np.concatenate([[0], np.cumsum(np.concatenate(counts))]).astype(np.int32)
    ci = rng.integers(0, K, rp[-1]).astype(np.int32)
    vv = np.where(rng.random(rp[-1]) < 0.1, 0.0, rng.uniform(-1, 1, rp[-1])).astype(np.float32)
    _say("convert window lengths", blk, K, M, ci.size)
    t = lambda a: torch.from_numpy(a).cuda()
    o = oracle.convert(rp, ci, vv, M, blk[0], blk[1])
    for _ in range(2):   # the second conversion works in memory that the first one has used
        plan = Plan(t(rp), t(ci), t(vv), M, blk[0], blk[1])
        _same(_arrays(plan), o)
        del plan


def test_device_conversion_many_long_windows(gpu):
    """More windows past the LDS classes than the key pass has grid rows: each
    keeps its own entries (the columns of neighbours overlap)."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    windows, K = 131, 40_000
    rng = np.random.default_rng(1)
    lens = rng.integers(16385, 17000, windows)
    M = windows * 16
    rp = np.zeros(M + 1, np.int64)
    for w, n in enumerate(lens):
        rp[w * 16 + 1:w * 16 + 17] = np.bincount(rng.integers(0, 16, n), minlength=16)
    rp = np.cumsum(rp).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(K, rp[r + 1] - rp[r], replace=False)) for r in range(M)]).astype(np.int32)
    vv = rng.uniform(-1, 1, ci.size).astype(np.float32)
    _say("convert long windows", windows, ci.size)
    t = lambda a: torch.from_numpy(a).cuda()
    _same(_arrays(Plan(t(rp), t(ci), t(vv), M)), oracle.convert(rp, ci, vv, M))


@pytest.mark.parametrize("lens", [(16385,), (300_000, 17000, 0, 1_048_577), (1_000_003,)])
def test_device_conversion_very_long_windows(gpu, lens):
    """Windows cut into segments over many workgroups: segments without a
    tile, duplicate columns across tile ends, explicit zeros."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    rng = np.random.default_rng(lens[0])
    M = 16 * len(lens) - 3
    counts = []
    for w, n in enumerate(lens):
        rows = min(16, M - 16 * w)
        counts.append(np.bincount(rng.integers(0, rows, n), minlength=rows))
    rp = np.concatenate([[0], np.cumsum(np.concatenate(counts))]).astype(np.int32)
    ci = rng.integers(0, 50_000, rp[-1]).astype(np.int32)      # unsorted, every column several times in a row
    vv = np.where(rng.random(rp[-1]) < 0.2, 0.0, rng.uniform(-1, 1, rp[-1])).astype(np.float32)
    _say("convert very long windows", lens)
    t = lambda a: torch.from_numpy(a).cuda()
    _same(_arrays(Plan(t(rp), t(ci), t(vv), M)), oracle.convert(rp, ci, vv, M))


@pytest.mark.parametrize("n", [3, 3000, 17000])   # windows sorted by 256 and 512 threads, and past LDS
def test_device_conversion_largest_column(gpu, n):
    """max_col is exact up to the largest column index: a dense operand must
    have more rows than it."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    ci = np.arange(n, dtype=np.int32)
    ci[-1] = 2**31 - 1
    _say("convert largest column", n)
    plan = Plan(*(torch.from_numpy(a).cuda() for a in (np.array([0, n], np.int32), ci, np.ones(n, np.float32))), 1)
    assert plan.max_col == 2**31 - 1


def test_device_conversion_rejects_malformed(gpu):
    import torch
    from mask_amd._capi import SrbcrsError
    from mask_amd.SRBCRSSpMM import Plan
    t = lambda a: torch.from_numpy(np.asarray(a)).cuda()
    with pytest.raises(SrbcrsError, match="non-decreasing"):
        Plan(t(np.array([0, 3, 1], np.int32)), t(np.array([0, 1, 2], np.int32)), t(np.ones(3, np.float32)), 2)
    with pytest.raises(SrbcrsError, match="non-decreasing"):
        Plan(t(np.array([0, 9], np.int32)), t(np.array([0, 1], np.int32)), t(np.ones(2, np.float32)), 1)
    with pytest.raises(SrbcrsError, match="negative"):
        Plan(t(np.array([0, 2], np.int32)), t(np.array([1, -4], np.int32)), t(np.ones(2, np.float32)), 1)


@pytest.mark.parametrize("name", ["convert_16x8_hand.json", "convert_32x32_hand.json"])
def test_device_conversion_matches_golden(gpu, name):
    """The device converter against the hand-derived fixtures."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    from tests.test_golden import arrays, load
    g = load(name)
    rp, ci, vv = arrays(g)
    t = lambda a: torch.from_numpy(a).cuda()
    _say("golden", name)
    got = _arrays(Plan(t(rp), t(ci), t(vv), g["num_nodes"], *g["blk"]))
    assert got["total"] == g["total"]
    for k in ("soff", "sidx", "block_partition", "edge_to_row", "edge_to_col"):
        assert got[k].tolist() == g[k], k
    assert got["val"].tobytes() == np.asarray(g["val"], np.float32).tobytes()


@pytest.mark.parametrize("a_operand", ["compact", "dense"])
@pytest.mark.parametrize("blk", [(16, 8), (32, 32)])
def test_spmm_exact_golden(gpu, blk, a_operand):
    """Power-of-two A times small-integer B: every sum is exact in fp32, so
    C must equal the fixture bit for bit."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    from tests.test_golden import arrays, load
    g = load("spmm_exact.json")
    rp, ci, vv = arrays(g)
    t = lambda a: torch.from_numpy(a).cuda()
    _say("exact spmm", blk, a_operand)
    plan = Plan(t(rp), t(ci), t(vv), g["num_nodes"], *blk)
    C = plan.run(t(np.asarray(g["B"], np.float32)), a_operand=a_operand).cpu().numpy()
    assert np.array_equal(C, np.asarray(g["C"], np.float32))
