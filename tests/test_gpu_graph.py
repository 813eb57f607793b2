"""The SpMM run path under HIP graph capture (torch.cuda.CUDAGraph): after
one eager run has sized the plan's buffers, a captured run replays correctly
many times, with eager work and new B values between the replays."""
from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import random_csr

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)


@pytest.mark.parametrize("policy", [("row", 0), ("split", 0), ("strict_lb", 5)])
def test_graph_replay_matches_eager(gpu, policy):
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    M, K, N = 613, 700, 128
    rp, ci, vv = random_csr(M, K, 0.02, 41, heavy_rows=3, heavy_len=650, empty_rows=0.1)
    t = lambda a: torch.from_numpy(a).cuda()
    plan = Plan(t(rp), t(ci), t(vv), M)
    plan.set_schedule(*policy)
    rng = np.random.default_rng(7)
    B = t(rng.uniform(-1, 1, (K, N)).astype(np.float32))
    C = torch.empty((M, N), device="cuda")
    _say("graph", policy)
    plan.run(B, C)                      # eager: sizes the partial buffer of split schedules
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            plan.run(B, C)
    torch.cuda.current_stream().wait_stream(s)
    for rep in range(4):
        B.copy_(t(rng.uniform(-1, 1, (K, N)).astype(np.float32)))
        C.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        got = C.clone()
        ref = plan.run(B)               # eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(got, ref), (policy, rep)


def test_graph_survives_partial_buffer_growth(gpu):
    """A run that needs a larger partial buffer (wider N, split schedule)
    after a graph was captured grows the buffer without freeing the old one,
    so replays of the earlier graph still write valid memory and stay
    correct; a schedule change keeps the captured task tables alive too."""
    import torch
    from mask_amd.SRBCRSSpMM import Plan
    M, K = 613, 700
    rp, ci, vv = random_csr(M, K, 0.02, 43, heavy_rows=3, heavy_len=650)
    t = lambda a: torch.from_numpy(a).cuda()
    plan = Plan(t(rp), t(ci), t(vv), M)
    plan.set_schedule("split", 3)
    rng = np.random.default_rng(9)
    B = t(rng.uniform(-1, 1, (K, 64)).astype(np.float32))
    C = torch.empty((M, 64), device="cuda")
    _say("graph growth")
    plan.run(B, C)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            plan.run(B, C)
    torch.cuda.current_stream().wait_stream(s)
    ref = plan.run(B).clone()
    wide = plan.run(t(rng.uniform(-1, 1, (K, 512)).astype(np.float32)))   # grows the partial buffer
    plan.set_schedule("strict_lb", 4)                                      # replaces the task tables
    plan.run(t(rng.uniform(-1, 1, (K, 512)).astype(np.float32)))
    torch.cuda.synchronize()
    for _ in range(3):
        C.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, ref)
    assert wide.shape == (M, 512)


def test_run_that_builds_its_stream_during_another_capture(gpu):
    """A default run on a stream that is not captured may allocate (its second
    run at a width builds the column sweep's stream) while another stream is
    captured: the capture stays valid, also where a conversion was refused in
    it."""
    import torch
    from mask_amd._capi import SrbcrsError
    from mask_amd.SRBCRSSpMM import Plan
    rng = np.random.default_rng(3)
    t = lambda a: torch.from_numpy(a).cuda()

    def csr(M, per):
        cols = np.sort(rng.integers(0, M, (M, per)), axis=1).astype(np.int32).ravel()
        return t(np.arange(M + 1, dtype=np.int32) * per), t(cols), t(rng.uniform(-1, 1, cols.size).astype(np.float32))

    small, large = csr(3000, 16), csr(60000, 16)
    p, q = Plan(*small, 3000), Plan(*large, 60000)
    B, C = torch.rand((3000, 64), device="cuda"), torch.empty((3000, 64), device="cuda")
    B2, C2 = torch.rand((60000, 128), device="cuda"), torch.empty((60000, 128), device="cuda")
    for _ in range(3):
        p.run(B, C)
    q.run(B2, C2)
    ref, ref2 = C.clone(), C2.clone()
    q.trim()                      # no kept memory: the stream's arrays come from hipMalloc
    other, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    _say("stream build during a capture")
    free = torch.cuda.mem_get_info()[0]
    with torch.cuda.graph(g):
        p.run(B, C)
        with torch.cuda.stream(other):
            q.run(B2, C2)
        with pytest.raises(SrbcrsError, match="capture"):
            Plan(*small, 3000)
    other.synchronize()
    assert free - torch.cuda.mem_get_info()[0] >= 8 * 60000 * 16
    assert torch.equal(C2, ref2)
    for _ in range(3):
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, ref)
        q.run(B2, C2)
        assert torch.equal(C2, ref2)
