"""The library's host code against a stand-in HIP runtime (tests/c/fake_hip.c,
no GPU): what it does when calls fail, under graph capture, and with device
memory over many calls.  Each test is a process of its own."""
from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)   # before the library: its HIP calls come here
import numpy as np
from mask_amd import _capi
L = _capi.lib()
fake.fake_live_bytes.restype = ctypes.c_size_t
fake.fake_launches.argtypes = [ctypes.c_char_p]
fake.fake_launches.restype = fake.fake_calls.restype = fake.fake_mallocs.restype = ctypes.c_long
launches = lambda part: fake.fake_launches(part.encode())
error = lambda: L.srbcrs_last_error().decode()

def d2h(data):
    data = np.ascontiguousarray(data)
    fake.fake_d2h(ctypes.c_size_t(data.nbytes), ctypes.c_void_p(data.ctypes.data))

def csr(M, K, per_row, seed=0):
    cols = np.sort(np.random.default_rng(seed).integers(0, K, (M, per_row)), axis=1).astype(np.int32).ravel()
    return (np.arange(M + 1, dtype=np.int32) * per_row, cols, np.ones(cols.size, np.float32))

def create(c, M, on_device):
    h = ctypes.c_void_p()
    rc = L.srbcrs_plan_create(*(a.ctypes.data for a in c), M, c[1].size, 16, 8, on_device, None, ctypes.byref(h))
    return rc, h

def head(blocks, stored, max_col):
    # what the conversion's kernels would have counted (struct Head)
    d2h(np.array([blocks, stored, 0, 0, 0, 0, max_col + 1, 0, 0, 0], np.uint32))

def sparse_plan(M, K, per_row):
    # a plan converted on the host, whose compact copy holds all its values
    c = csr(M, K, per_row)
    d2h(np.array([0, c[1].size], np.uint32))
    rc, h = create(c, M, 0)
    assert rc == 0, error()
    fake.fake_d2h(ctypes.c_size_t(0), None)
    return h

def run(h, M, K, N, B=np.zeros(1 << 22, np.float32), C=np.zeros(1 << 22, np.float32)):
    assert K * N <= B.size and M * N <= C.size
    align = lambda a: (a.ctypes.data + 15) // 16 * 16
    return L.srbcrs_run(h, align(B), K, N, N, align(C), N, M, None)
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["gcc", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", str(so),
                    str(ROOT / "tests" / "c" / "fake_hip.c")], check=True)
    return so


def _run(fake_hip, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, str(fake_hip)], cwd=ROOT, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout[-1000:] + r.stderr[-2000:]


# the conversion's synchronisations: after the window scan, and at its end
@pytest.mark.parametrize("good_syncs", [0, 1])
def test_conversion_reports_a_failure_of_its_kernels(fake_hip, good_syncs):
    """An error that shows only when the stream is waited for is the call's
    result, and none of the memory is kept for another conversion."""
    _run(fake_hip, f"""
c = csr(320, 500, 5)
head(900, c[1].size, 499)
fake.fake_fail_sync({good_syncs})
rc, h = create(c, 320, 1)
assert launches("k_blocks") == {good_syncs}
assert rc == _capi.SRBCRS_EHIP and not h.value, (rc, error())
assert fake.fake_live_blocks() == 0
fake.fake_fail_sync(-1)
rc, h = create(c, 320, 1)
assert rc == 0, error()
""")


def test_conversion_under_capture_is_refused_before_any_call(fake_hip):
    """Also with kept memory at hand: nothing is recorded into the graph."""
    _run(fake_hip, """
c = csr(320, 500, 5)
head(900, c[1].size, 499)
rc, h = create(c, 320, 1)
assert rc == 0, error()
L.srbcrs_plan_destroy(h)
calls, mallocs = fake.fake_calls(), fake.fake_mallocs()
fake.fake_capture(1)
rc, h = create(c, 320, 1)
assert rc == _capi.SRBCRS_ENOMEM and "capture" in error(), (rc, error())
assert (fake.fake_calls(), fake.fake_mallocs()) == (calls, mallocs)
fake.fake_capture(0)
assert create(c, 320, 1)[0] == 0, error()
""")


def test_a_sweep_stream_that_could_not_be_built_is_tried_again(fake_hip):
    """A shortage of memory sends the run to the block kernels and is not
    remembered for good; one that lasts is not met on every run."""
    _run(fake_hip, """
M = K = 4096
h = sparse_plan(M, K, 20)
assert run(h, M, K, 64) == 0 and launches("spmm_colsweep") == 0
fake.fake_fail_malloc(1, 2)     # the flags are allocated, the stream's arrays are not
assert run(h, M, K, 64) == 0, error()
assert launches("spmm_colsweep") == 0 and launches("spmm_stream") == 2
for _ in range(3):
    assert run(h, M, K, 64) == 0, error()
assert launches("spmm_colsweep") >= 1
h = sparse_plan(M, K, 20)
assert run(h, M, K, 64) == 0
before = fake.fake_mallocs()
fake.fake_fail_malloc(0, 1 << 30)
for _ in range(500):
    assert run(h, M, K, 64) == 0, error()
assert fake.fake_mallocs() - before < 500   # under one a run; an attempt makes 32
""")


def test_sweep_streams_are_bounded_and_trimmed(fake_hip):
    """However many widths run, the streams of one schedule hold at most the
    size of the block values; trim frees those of other schedules that no
    captured run holds."""
    _run(fake_hip, """
M = K = 65536
big = dict(B=np.zeros(512 * K + 8, np.float32), C=np.zeros(512 * M + 8, np.float32))
h = sparse_plan(M, K, 16)
d = _capi.PlanDesc()
L.srbcrs_plan_get(h, ctypes.byref(d))
entries = M * 16 * 5 // 4
d2h(np.array([entries, 0], np.uint64))                              # a list stream
d2h(np.array([entries, 0, M * 16, M * 16], np.uint64))              # a phase stream
trim = lambda: L.srbcrs_plan_trim(h, None)
live = lambda: (trim(), fake.fake_live_bytes())[1]
base = live()
for N in range(32, 513, 16):
    for i in range(3):
        assert run(h, M, K, N, **big) == 0, error()
    assert launches("spmm_stream") <= 2 * N // 16
    assert launches("spmm_colsweep") + launches("spmm_phasesweep") >= N // 16 - 1   # at least the last of the three
    assert live() - base <= d.total_blocks * 512 + 8 * entries
row = live()
assert row - base > 3 * 8 * entries
def schedule(p, q):
    assert L.srbcrs_plan_set_schedule(h, p, q) == 0, error()
one = 8 * entries   # and its padding and places
def split(p):
    schedule(b"split", p)
    assert run(h, M, K, 512, **big) == 0, error()   # the block kernels; the partial tiles are allocated
    base = live()
    assert run(h, M, K, 512, **big) == 0, error()
    assert one < live() - base < 2 * one
    return base
no_streams = split(7)
fake.fake_capture(1)
assert run(h, M, K, 512, **big) == 0, error()
fake.fake_capture(0)
assert one // 2 < split(9) - no_streams < 2 * one   # the stream that the capture holds
schedule(b"row", 0)
assert one // 2 < live() - no_streams < 2 * one     # the other is gone
for N in (64, 512):   # built again, by the second run at the latest
    assert run(h, M, K, N, **big) == 0, error()
    n = launches("spmm_colsweep") + launches("spmm_phasesweep")
    assert run(h, M, K, N, **big) == 0, error()
    assert launches("spmm_colsweep") + launches("spmm_phasesweep") == n + 1
L.srbcrs_plan_destroy(h)
""")


def test_kept_memory_is_bounded_in_waste_and_given_back(fake_hip):
    """A large block is at most a thirty-second more than asked for, what a run
    allocates is just that, and with no plan left all memory can be released."""
    _run(fake_hip, """
M, N = 300000, 512
c = csr(M, 20000, 1)
blocks = 131073
head(blocks, c[1].size, 19999)
calls = []
rc, h = create(c, M, 1)
assert rc == 0, error()
d = _capi.PlanDesc()
L.srbcrs_plan_get(h, ctypes.byref(d))
assert d.total_blocks == blocks
L.srbcrs_plan_trim(h, None)
own = 4 * (M // 16 + 2) + 8 * c[1].size + 4 * M // 16 + blocks * (512 + 32 + 32) + 4 * c[1].size
assert own <= fake.fake_live_bytes() < own * 33 // 32 + (1 << 20)
L.srbcrs_plan_destroy(h)
assert fake.fake_live_bytes() >= own
assert L.srbcrs_release_memory() == 0 and fake.fake_live_bytes() == 0
fake.fake_fail_malloc(0, 1 << 30)
rc, h = create(c, M, 1)
assert rc == _capi.SRBCRS_ENOMEM and "out of memory" in error(), error()
""")


def test_kept_memory_of_many_sizes_costs_no_time(fake_hip):
    """A conversion takes what it took before 400 graphs of other sizes were
    dropped, whose arrays are all kept."""
    _run(fake_hip, """
import time
c = csr(64, 500, 5)
def once():
    head(200, c[1].size, 499)
    rc, h = create(c, 64, 1)
    assert rc == 0, error()
    L.srbcrs_plan_destroy(h)
def best():
    times = []
    for _ in range(200):
        t = time.perf_counter()
        once()
        times.append(time.perf_counter() - t)
    return sorted(times)[20]
before = best()
plans = []
for i in range(400):
    o = csr(640 + 48 * i, 500, 5)
    head(200 + 7 * i, o[1].size, 499)
    rc, h = create(o, 640 + 48 * i, 1)
    assert rc == 0, error()
    plans.append(h)
for h in plans:
    L.srbcrs_plan_destroy(h)
assert fake.fake_live_blocks() > 2000
after = best()
print(before, after)
assert after < 1.5 * before + 2e-5, (before, after)
""")


# (M, K, values a row, N, schedule, span of a window's columns, whether the second run is a sweep):
# both sides of the dispatch rules
@pytest.mark.parametrize("M,K,per_row,N,schedule,span,sweep", [
    (20000, 300000, 16, 256, "row:0", 0, False), (20000, 60000, 10, 256, "row:0", 0, True),   # too few rows for lists
    (60000, 300000, 16, 64, "row:0", 0, False), (60000, 100000, 16, 64, "row:0", 0, True),
    (2000, 100000, 40, 256, "row:0", 0, True), (20000, 300000, 10, 224, "row:0", 0, True),
    (200000, 300000, 4, 256, "row:0", 0, False), (200000, 300000, 12, 256, "row:0", 0, True),  # very short rows
    (100000, 400000, 7, 256, "row:0", 0, False),                                             # few values a column
    (60000, 100000, 19, 16, "row:0", 0, False), (60000, 100000, 20, 16, "row:0", 0, True),    # 16 columns
    (200000, 10000, 12, 16, "row:0", 0, True),
    (200000, 200000, 16, 128, "row:0", 20000, False), (200000, 200000, 16, 128, "row:0", 30000, True),   # local, many rows
    (60000, 60000, 16, 128, "row:0", 400, True), (200000, 200000, 16, 48, "row:0", 400, True),
    (60000, 60000, 3, 256, "row:0", 400, False), (60000, 60000, 5, 256, "row:0", 400, True),  # reuse 1 of short local rows
    (4096, 4096, 20, 64, "row:0", 0, True), (4096, 4096, 20, 64, "split:16", 0, False),       # small: long tasks only
    (4096, 4096, 20, 64, "split:31", 0, False), (4096, 4096, 20, 64, "split:32", 0, True),
    (20000, 20000, 20, 64, "split:8", 0, False), (20000, 20000, 20, 64, "split:9", 0, True),  # short tasks
    (20000, 20000, 20, 128, "split:8", 0, True), (1000, 1000, 4, 64, "row:0", 0, False),
])
def test_which_runs_are_sweeps(fake_hip, M, K, per_row, N, schedule, span, sweep):
    _run(fake_hip, f"""
M, K, N = {M}, {K}, {N}
big = dict(B=np.zeros(N * K + 8, np.float32), C=np.zeros(N * M + 8, np.float32))
h = sparse_plan(M, K, {per_row})
windows = (M + 15) // 16
d2h(np.array([windows * {span}, windows if {span} else 0, 0], np.uint64))            # the window spans
d2h(np.array([M * {per_row} * 5 // 4, 0], np.uint64))                                # a list stream
d2h(np.array([M * {per_row} * 5 // 4, 0, M * {per_row}, M * {per_row}], np.uint64))  # a phase stream
policy, param = "{schedule}".split(":")
assert L.srbcrs_plan_set_schedule(h, policy.encode(), int(param)) == 0, error()
for i in range(3):
    assert run(h, M, K, N, **big) == 0, error()
assert launches("spmm_colsweep") + launches("spmm_phasesweep") == 2 * {int(sweep)}
assert launches("spmm_stream") == 3 - 2 * {int(sweep)}
""")


def test_windows_of_unlike_length_keep_the_sweep(fake_hip):
    """Rows that would stay with the block kernels, but for a window 20 times as long."""
    for heavy, sweep in ((10, 0), (4000, 2)):
        _run(fake_hip, f"""
M, K, N = 60000, 60000, 16
rp, cols, vals = csr(M, K, 10)
cols = np.concatenate([np.sort(np.random.default_rng(1).choice(K, {heavy}, replace=False)).astype(np.int32), cols[10:]])
rp[1:] += {heavy} - 10
vals = np.ones(cols.size, np.float32)
d2h(np.array([0, cols.size], np.uint32))
rc, h = create((rp, cols, vals), M, 0)
assert rc == 0, error()
d2h(np.array([M * 13, 0], np.uint64))
d2h(np.array([M * 13, 0, M * 10, M * 10], np.uint64))
for i in range(3):
    assert run(h, M, K, N) == 0, error()
assert launches("spmm_colsweep") + launches("spmm_phasesweep") == {sweep}
""")
