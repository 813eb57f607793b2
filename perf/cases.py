"""The work a user of this framework has it do, as cases that can be timed and checked.

Each case is one call (or one short sequence of calls) through the public entry points: the
drop-in module ``mask_amd.SRBCRSSpMM`` (preprocess, run, CSR kernel), its ``Plan`` objects, the
GCN bridge ``mask_amd.external_backend_spmm`` and the GCN on top of it (``mask_amd.gcn``).

``op`` of a case:
  run       SpMM through ``Plan.run`` with no knobs, the schedule ``auto`` that the drop-in picks
  dropin    SpMM through ``run_SRBCRS_16x8`` on arrays that ``preprocess_gpu_16x8`` gave before
  sweep     SpMM through the nonzero sweep (``Plan.run(grid_order=5)``), the vector path that a
            caller opts into for low block density
  relu      relu(A B) in one call, into a buffer that the caller keeps
  csr       the CSR kernel of the fallback, on the caller's CSR arrays
  bridge    one forward SpMM through the GCN bridge at a feature width that may need padding
  layer     the GCN aggregation with autograd: forward A h, backward A^T g
  train     a GCN training step: forward, loss, backward
  convert   preprocess of a new graph: CSR to SR-BCRS, with the edge maps
  fresh     a graph used once (a sampled mini-batch): preprocess, one SpMM, dropped

``graph`` of a case:
  uniform   ``per_row`` distinct random columns in each of M rows, K columns
  bernoulli M x K, every entry with probability ``per_row / K`` (rows of unequal length)
  banded    full 16x8 blocks near the diagonal (M / 16 block rows, each of 9 kept with
            probability 0.7), K = M
  rmat      a power-law graph of M nodes and about ``M * per_row`` directed edges, symmetrised,
            with self loops and the values D^-1/2 (A + I) D^-1/2, K = M
"""
from __future__ import annotations

import math
import weakref

import torch

from mask_amd import SRBCRSSpMM
from mask_amd.external_backend_spmm import SRBCRSBackend, reset_backend_state
from mask_amd.gcn import GCN, Graph, aggregate

CLASSES = 64                # output width of the training step's GCN
MAX_GATHER = 40_000_000_000   # bytes of dense rows that a drawn case's SpMM refers to, at most


def listed():
    return [
        # the smallest SpMM: a 4096-node graph at one 64-wide feature tile; the call and its latency count
        dict(name="small-n64", op="dropin", graph="bernoulli", M=4096, K=4096, per_row=20, N=64),
        # the SpMM benchmark's uniform matrix as a drop-in user runs it, without knobs
        dict(name="uniform-n512", op="dropin", graph="uniform", M=65536, K=65536, per_row=16, N=512),
        # the same matrix as the benchmark's headline runs it: the opt-in for low block density
        dict(name="uniform-n512-sweep", op="sweep", graph="uniform", M=65536, K=65536, per_row=16, N=512),
        # full blocks near the diagonal, as a discretised PDE or a blocked factor has them; the largest output
        dict(name="banded-n512", op="run", graph="banded", M=524288, K=524288, per_row=0, N=512),
        # the largest power-law graph, heavy-tailed rows (split schedule)
        dict(name="rmat-n512", op="run", graph="rmat", M=1 << 20, K=1 << 20, per_row=16, N=512),
        # the hidden layer's aggregation of the GCN workload with its backward, on a social-network-sized graph
        dict(name="gcn-layer-n256", op="layer", graph="rmat", M=232965, K=232965, per_row=25, N=256),
        # a GCN's last layer: the class count is no multiple of any tile, the node count of no window
        dict(name="gcn-out-n41", op="bridge", graph="rmat", M=116483, K=116483, per_row=12, N=41),
        # a hidden layer at inference with its activation fused, rectangular (a bipartite block of a sampled graph)
        dict(name="relu-n128", op="relu", graph="uniform", M=100003, K=30011, per_row=10, N=128),
        # the whole model: a two-layer GCN training step
        dict(name="train-512-256-64", op="train", graph="rmat", M=58241, K=58241, per_row=25, N=256),
        # loading a graph: the conversion of the GCN workload's adjacency
        dict(name="convert-large", op="convert", graph="rmat", M=232965, K=232965, per_row=25, N=0),
        # a sampled mini-batch: converted, used once, dropped
        dict(name="fresh-n128", op="fresh", graph="uniform", M=8191, K=20011, per_row=12, N=128),
        # the fallback kernel, on rows of unequal length
        dict(name="csr-n256", op="csr", graph="bernoulli", M=50021, K=65536, per_row=24, N=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["run", "dropin", "sweep", "relu", "csr", "bridge", "layer", "train", "convert", "fresh"])
    if op == "train":
        graph = "rmat"
    elif op in ("layer", "bridge"):
        graph = rng.choice(["rmat", "rmat", "bernoulli"])
    elif op in ("sweep", "csr", "fresh"):
        graph = rng.choice(["uniform", "bernoulli"])
    else:
        graph = rng.choice(["uniform", "bernoulli", "banded", "rmat"])
    top = {"train": 60000, "fresh": 40000, "convert": 250000, "layer": 250000}.get(op, 400000)
    M = _log_int(rng, 1000, top)
    square = graph in ("banded", "rmat") or op in ("layer", "train")
    if graph == "banded":
        M = max(16, M // 16 * 16 - rng.choice([0, 0, 5]))
    K = M if square else _log_int(rng, 1000, top)
    per_row = 0 if graph == "banded" else _log_int(rng, 4, 48)
    if op == "convert":
        N = 0
    elif op == "train":
        N = rng.choice([64, 96, 128, 256])
    elif op in ("bridge", "layer"):
        N = rng.choice([16, 41, 64, 100, 128, 200, 256, 300])
    elif op == "sweep":
        N = 64 * rng.choice([1, 2, 3, 4, 6, 8])
    elif op == "csr":
        N = rng.choice([17, 64, 100, 128, 256, 320, 512])
    else:
        N = 16 * rng.choice([1, 2, 3, 4, 6, 7, 8, 12, 16, 20, 24, 32])
    case = dict(op=op, graph=graph, M=M, K=K, per_row=per_row, N=N)
    while _nnz(case) * max(N, 64) * 4 > MAX_GATHER and case["per_row"] > 4:
        case["per_row"] = max(4, case["per_row"] // 2)
    return case


def _nnz(case):
    """About how many values the matrix stores."""
    if case["graph"] == "banded":
        return int(math.ceil(case["M"] / 16) * 9 * 0.7 * 128)
    if case["graph"] == "rmat":
        return case["M"] * (2 * case["per_row"] + 1)
    return case["M"] * min(case["per_row"], case["K"])


# ---- inputs ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _csr(rows, cols, M):
    rowptr = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(torch.bincount(rows, minlength=M), 0)
    return rowptr.to(torch.int32), cols.to(torch.int32)


def _distinct(key, K, M):
    key = torch.unique(key)   # sorted: by row, then column
    return _csr(torch.div(key, K, rounding_mode="floor"), key % K, M)


def _uniform(M, K, per_row, g):
    per_row = min(per_row, K)
    cols = torch.randint(0, K, (M, per_row), generator=g, device="cuda").sort(dim=1).values
    for _ in range(100):   # redraw the rows that hold a column twice
        bad = (cols[:, 1:] == cols[:, :-1]).any(dim=1).nonzero().flatten()
        if bad.numel() == 0:
            break
        cols[bad] = torch.randint(0, K, (bad.numel(), per_row), generator=g, device="cuda").sort(dim=1).values
    rowptr = torch.arange(M + 1, device="cuda") * per_row
    return rowptr.to(torch.int32), cols.reshape(-1).to(torch.int32)


def _bernoulli(M, K, per_row, g):
    n = torch.poisson(torch.full((1,), float(M * per_row), device="cuda"), generator=g)
    key = torch.randint(0, M * K, (max(1, int(n.item())),), generator=g, device="cuda")
    return _distinct(key, K, M)


def _banded(M, g):
    block_rows = (M + 15) // 16
    i = torch.arange(block_rows, device="cuda")[:, None]
    j = 2 * i + torch.arange(-4, 5, device="cuda")[None, :]
    keep = (j >= 0) & (8 * j + 8 <= M) & (torch.rand(j.shape, generator=g, device="cuda") < 0.7)
    bj = j[keep]                                   # in block-row order, columns ascending
    count = keep.sum(dim=1)
    first = torch.cumsum(count, 0) - count
    rows = torch.arange(M, device="cuda")
    length = 8 * count[rows // 16]
    rowptr = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(length, 0)
    row = torch.repeat_interleave(rows, length)
    pos = torch.arange(row.numel(), device="cuda") - rowptr[row]
    cols = bj[first[row // 16] + pos // 8] * 8 + pos % 8
    return rowptr.to(torch.int32), cols.to(torch.int32)


def _rmat(n, per_row, g):
    scale = max(1, (n - 1).bit_length())
    need, parts = n * per_row, []
    while need > 0:
        src = torch.zeros(need, dtype=torch.int64, device="cuda")
        dst = torch.zeros(need, dtype=torch.int64, device="cuda")
        for level in range(scale):   # quadrant probabilities 0.5, 1/6, 1/6, 1/6
            u = torch.rand(need, generator=g, device="cuda")
            down = u >= 2 / 3
            right = ((u >= 0.5) & (u < 2 / 3)) | (u >= 5 / 6)
            src |= down.to(torch.int64) << level
            dst |= right.to(torch.int64) << level
        ok = (src < n) & (dst < n)
        parts.append((src[ok], dst[ok]))
        need -= int(ok.sum().item())
    src = torch.cat([p[0] for p in parts])
    dst = torch.cat([p[1] for p in parts])
    loops = torch.arange(n, device="cuda")
    return _distinct(torch.cat([src * n + dst, dst * n + src, loops * n + loops]), n, n)


def _row_ids(rowptr):
    return torch.repeat_interleave(torch.arange(rowptr.numel() - 1, device="cuda"), (rowptr[1:] - rowptr[:-1]).long())


def _matrix(case, g):
    M, K = case["M"], case["K"]
    if case["graph"] == "rmat":
        rowptr, colind = _rmat(M, case["per_row"], g)
        inv = (rowptr[1:] - rowptr[:-1]).double().rsqrt()
        values = (inv[_row_ids(rowptr)] * inv[colind.long()]).float()
        return rowptr, colind, values
    if case["graph"] == "uniform":
        rowptr, colind = _uniform(M, K, case["per_row"], g)
    elif case["graph"] == "bernoulli":
        rowptr, colind = _bernoulli(M, K, case["per_row"], g)
    else:
        rowptr, colind = _banded(M, g)
    if case["graph"] == "banded":
        values = torch.randn(colind.numel(), generator=g, device="cuda")
    else:
        values = torch.rand(colind.numel(), generator=g, device="cuda") * 2 - 1
    return rowptr, colind, values


def _transpose(csr, K):
    rowptr, colind, values = csr
    order = torch.sort(colind.long(), stable=True).indices
    t_rowptr, t_colind = _csr(colind.long()[order], _row_ids(rowptr)[order], K)
    return t_rowptr, t_colind, values[order].contiguous()


def _inputs(case, seed):
    """The CSR matrix and the dense operand (and, for the layers, the gradient that comes back)."""
    g = _gen(seed)
    csr = _matrix(case, g)
    extra = {}
    if case["op"] == "train":
        extra["x"] = torch.randn((case["M"], 2 * case["N"]), generator=g, device="cuda")
        extra["y"] = torch.randint(0, CLASSES, (case["M"],), generator=g, device="cuda")
    elif case["N"]:
        shape = (case["K"], case["N"])
        normal = case["graph"] in ("rmat", "banded")
        extra["dense"] = (torch.randn(shape, generator=g, device="cuda") if normal
                          else torch.rand(shape, generator=g, device="cuda") * 2 - 1)
        if case["op"] == "layer":
            extra["grad"] = torch.randn((case["M"], case["N"]), generator=g, device="cuda")
    return csr, extra


class _State(dict):
    """A dict that a weak set can hold."""
    __hash__ = object.__hash__
    __eq__ = object.__eq__


_alive = weakref.WeakSet()


def _most_edges(case):
    """A bound on the stored values, whatever the seed (of a Poisson count, 8 deviations up)."""
    n = _nnz(case)
    if case["graph"] == "bernoulli":
        n += 8 * math.isqrt(n) + 64
    return n if case["graph"] != "banded" else (case["M"] + 15) // 16 * 9 * 128


def _edge_buffers(case, n):
    """The output buffers that preprocess fills: block_partition, edge_to_col, edge_to_row."""
    i32 = dict(dtype=torch.int32, device="cuda")
    return torch.zeros((case["M"] + 15) // 16, **i32), torch.zeros(n, **i32), torch.zeros(n, **i32)


def _preprocess(csr, M, buffers):
    return SRBCRSSpMM.preprocess_gpu_16x8(csr[1], csr[0], csr[2], M, 16, 8, *buffers)


def prepare(case, seed):
    if len(_alive) == 0:   # a program that drops its graphs also drops the conversions the modules hold
        reset_backend_state()
        SRBCRSSpMM.clear_cache()
    s = _State(case=case)
    csr, extra = _inputs(case, seed)
    s.update(csr=csr, **extra)
    op, M = case["op"], case["M"]
    if op in ("run", "sweep", "relu"):
        s["plan"] = SRBCRSSpMM.Plan(*csr, M)
        if op != "sweep":
            s["plan"].set_schedule("auto")
        if op == "relu":
            s["out"] = torch.empty((M, case["N"]), device="cuda")
    elif op == "dropin":
        s["arrays"] = _preprocess(csr, M, _edge_buffers(case, csr[1].numel()))
    elif op == "bridge":
        s["backend"] = SRBCRSBackend("16x8")
    elif op in ("layer", "train"):
        s["backend"] = SRBCRSBackend("16x8")
        s["graph"] = Graph("graph", M, csr[1].numel(), csr, _transpose(csr, case["K"]), s.get("x"))
        if op == "layer":
            s["h"] = s["dense"].clone().requires_grad_(True)
        else:
            s["model"] = GCN((2 * case["N"], case["N"], CLASSES), spmm=s["backend"].run, seed=seed).to("cuda")
    elif op in ("convert", "fresh"):   # buffers kept from graph to graph, large enough for any of them
        s["buffers"] = _edge_buffers(case, _most_edges(case))
        s["index"] = torch.zeros(_most_edges(case) + 8 * ((M + 15) // 16), dtype=torch.int32, device="cuda")
    _alive.add(s)
    return s


# ---- one pass ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    op, M = case["op"], case["M"]
    csr = s["csr"]
    if op == "run":
        return s["plan"].run(s["dense"])
    if op == "sweep":
        return s["plan"].run(s["dense"], grid_order=5)
    if op == "relu":
        return s["plan"].run(s["dense"], s["out"], relu=True)
    if op == "csr":
        return SRBCRSSpMM.csr_spmm(*csr, s["dense"], M)
    if op == "dropin":
        rwo, _rowid, tile_id, toff, a2x, _total = s["arrays"]
        return SRBCRSSpMM.run_SRBCRS_16x8(s["dense"], rwo, tile_id, toff, a2x, M, csr[1].numel(), "")[0]
    if op == "bridge":
        return s["backend"].run(*csr, s["dense"], M, case["N"], M)
    if op == "layer":
        s["h"].grad = None
        out = aggregate(s["graph"], s["h"], s["backend"].run)
        out.backward(s["grad"])
        return out.detach(), s["h"].grad
    if op == "train":
        model = s["model"]
        model.zero_grad()
        logp = model(s["graph"])
        loss = torch.nn.functional.nll_loss(logp, s["y"])
        loss.backward()
        return logp.detach(), loss.detach(), [p.grad for p in model.parameters()]
    rwo, _rowid, tile_id, toff, a2x, total = _preprocess(csr, M, s["buffers"])
    s["index"][:tile_id.numel()].copy_(tile_id)
    out = (rwo, s["index"], total, *s["buffers"])
    if op == "fresh":
        out += (SRBCRSSpMM.run_SRBCRS_16x8(s["dense"], rwo, tile_id, toff, a2x, M, csr[1].numel(), "")[0],)
    SRBCRSSpMM.clear_cache()
    return out


# ---- what a pass needs, and what it gives -----------------------------------------------------

def work(case):
    """Bytes and operations of one pass: the CSR matrix, the dense operand once, the result once."""
    nnz, M, K, N = _nnz(case), case["M"], case["K"], case["N"]
    a = 8 * nnz + 4 * (M + 1)
    spmm = dict(bytes=a + 4 * N * (M + K), flops=2 * nnz * N)
    conversion = a + 4 * (2 * nnz + M // 16) + 8 * nnz   # CSR in; edge maps, index and value arrays out
    if case["op"] == "layer":
        return dict(bytes=2 * spmm["bytes"], flops=2 * spmm["flops"])
    if case["op"] == "train":
        c, f = CLASSES, 2 * N
        gemms = 2 * M * (2 * f * N + 3 * N * c)   # X W1, dW1; H W2, dW2, dH
        return dict(bytes=4 * a + 4 * M * (2 * f + 6 * N + 6 * c), flops=4 * nnz * (N + c) + gemms)
    if case["op"] == "convert":
        return dict(bytes=conversion, flops=0)
    if case["op"] == "fresh":
        return dict(bytes=conversion + spmm["bytes"], flops=spmm["flops"])
    return spmm


def tolerance(case):
    """fp32 products and sums, measured up to 1.3e-7 from the same in 64 bits; two correct orders of
    summation differ by up to about twice that.  In the training step a hidden unit whose sum is
    within rounding of zero passes relu in one order and not in another, which changes the first
    layer's gradient by about one in the square root of its terms (4.2e-4 measured)."""
    if case["op"] == "convert":
        return "exact"
    if case["op"] == "train":
        return dict(rel=2e-3, max=5e-2)
    return dict(rel=1e-6, max=4e-5)


# ---- the same in 64 bits ------------------------------------------------------------------------

def _product(csr, dense, K):
    """A @ dense in 64 bits."""
    rowptr, colind, values = csr
    a = torch.sparse_csr_tensor(rowptr.long(), colind.long(), values.double(), size=(rowptr.numel() - 1, K))
    parts = [torch.sparse.mm(a, dense[:, c:c + 64].double().contiguous()) for c in range(0, dense.shape[1], 64)]
    return torch.cat(parts, dim=1)


def exact(case, seed):
    op = case["op"]
    if op == "convert":
        return None
    csr, extra = _inputs(case, seed)
    K = case["K"]
    if op == "layer":
        return _product(csr, extra["dense"], K), _product(_transpose(csr, K), extra["grad"], case["M"])
    if op == "train":
        at = _transpose(csr, K)
        weights = GCN((2 * case["N"], case["N"], CLASSES), seed=seed).weights
        w1, w2 = (w.detach().to("cuda").double() for w in weights)
        x, y = extra["x"].double(), extra["y"]
        pre = _product(csr, x @ w1, K)
        h = torch.relu(pre)
        z = _product(csr, h @ w2, K)
        logp = torch.log_softmax(z, dim=1)
        loss = torch.nn.functional.nll_loss(logp, y)
        dz = logp.exp()
        dz[torch.arange(y.numel(), device="cuda"), y] -= 1
        dq = _product(at, dz / y.numel(), case["M"])
        dp = _product(at, (dq @ w2.t()) * (pre > 0), case["M"])
        return logp, loss, [x.t() @ dp, h.t() @ dq]
    c = _product(csr, extra["dense"], K)
    if op == "fresh":
        return (None,) * 6 + (c,)
    return torch.relu(c) if op == "relu" else c
