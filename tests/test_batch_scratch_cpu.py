"""Scratch of the batched decode (9..63 tokens of row-split weights) in the
host code: runtime.cpp linked to a recording stand-in for HIP and the kernel
launches (tests/c/host_stub.cpp), so every launch's scratch pointers, and
every allocation, free and wait of a call are seen without a GPU.

One to eight tokens of a row-split weight need no scratch, and neither did
batches launched eight tokens at a time: a HIP graph of them can be replayed
on any stream beside any other work.  The batch keeps that by never being
captured.
"""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "qwen38-in-c_amd", "csrc")
S, T, U = 0x1000, 0x2000, 0x3000   # streams


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("g++ and the HIP headers needed")
    so = str(tmp_path_factory.mktemp("stub") / "libhoststub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-fPIC", "-shared", "-fvisibility=hidden",
                    "-Wl,-Bsymbolic", "-Wl,--no-undefined", "-o", so, os.path.join(ROOT, "tests", "c", "host_stub.cpp"),
                    os.path.join(CSRC, "runtime.cpp"), os.path.join(CSRC, "safetensors.cpp"), "-lpthread", "-ldl"],
                   check=True)
    return so


class Lib:
    """The library over the stand-in; addresses in place of device tensors."""

    def __init__(self, path):
        import q35mm
        self.lib = q35mm._load(path)
        self.lib.stub_log.restype = C.c_char_p
        self.lib.stub_capture.argtypes = [C.c_void_p, C.c_int]
        self.lib.stub_fail_malloc.argtypes = [C.c_size_t]
        self.x, self.y = 1 << 40, 1 << 41
        assert self.lib.q35mm_init(0) == 0
        self.take()

    def weight(self, rows, cols, wide=False):
        W = np.zeros((rows, cols), np.uint8)
        sc = np.full(((rows + 127) // 128, (cols + 127) // 128), 0x3F80, np.uint16)
        if wide:
            sc[0, 0], sc[0, 1] = 0x6F80, 0x3380     # 2^96 and 2^-24: beyond the GEMM
        w = C.c_void_p()
        p8, p16 = C.POINTER(C.c_uint8), C.POINTER(C.c_uint16)
        assert self.lib.q35mm_weight_create(W.ctypes.data_as(p8), sc.ctypes.data_as(p16), rows, cols, C.byref(w)) == 0
        self.take()
        return w

    def take(self):
        """The recorded lines since the last take: (kind, {key: value})."""
        lines = self.lib.stub_log().decode().splitlines()
        self.lib.stub_clear()
        return [(ln.split()[0], dict(f.split("=") for f in ln.split() if "=" in f), ln) for ln in lines]

    def matmul(self, w, m, st):
        return self.lib.q35mm_matmul(w, m, self.x, self.y, st), self.take()

    def mlp(self, ws, m, st):
        return self.lib.q35mm_mlp(*ws, self.x, 1e-6, m, self.x, st), self.take()

    def capture(self, st, on=True):
        self.lib.stub_capture(st, int(on))


@pytest.fixture
def lib(stub_path):
    lb = Lib(stub_path)
    yield lb
    lb.lib.stub_fail_malloc(C.c_size_t(-1))
    for s in (None, S, T, U):
        lb.capture(s, False)
    lb.lib.q35mm_shutdown()
    lb.take()


def kinds(rec):
    return [r[0] for r in rec]


def pointers(rec):
    """Scratch addresses a call's launches carry."""
    return {v for _, f, _ in rec for k, v in f.items() if k in ("xs", "xf", "ws", "xb", "cnt") and v != "(nil)"}


def test_eager_batch(lib):
    """What the other tests build on: outside capture 24 tokens are a batch."""
    w = lib.weight(300, 1024)
    rc, rec = lib.matmul(w, 24, S)
    assert rc == 0 and [k for k in kinds(rec) if k in ("split", "batch", "rows")] == ["split", "batch"]


@pytest.mark.parametrize("m", [9, 24, 63])
def test_captured_matmul_carries_no_scratch(lib, m):
    """A stream with scratch of its own, warmed at the same size: two graphs
    of the call hold no memory in common, so they may be replayed at once."""
    w = lib.weight(300, 5120)
    assert lib.matmul(w, m, S)[0] == 0
    assert lib.matmul(w, 512, S)[0] == 0
    lib.capture(S)
    for _ in range(2):
        rc, rec = lib.matmul(w, m, S)
        assert rc == 0 and kinds(rec) == ["rows"] * ((m + 7) // 8) and not pointers(rec)


@pytest.mark.parametrize("m", [9, 24])
def test_captured_mlp_carries_only_its_workspace(lib, m):
    """The MLP block's graph holds the block's own intermediates, as it did
    in groups of eight tokens, and none of the scratch matmuls use."""
    ws = [lib.weight(1664, 5120), lib.weight(1664, 5120), lib.weight(5120, 1664)]
    assert lib.mlp(ws, m, S)[0] == 0
    lib.capture(S)
    rc, rec = lib.mlp(ws, m, S)
    n = (m + 7) // 8
    assert rc == 0 and kinds(rec) == ["rmsnorm"] + ["pair"] * n + ["rows"] * n and not pointers(rec)


@pytest.mark.parametrize("m", [9, 24, 63])
def test_noalloc_uses_no_shared_scratch(lib, m):
    """Every stream's allocation-free calls share one fixed array; row-split
    weights use none of it, so these calls may overlap on two streams."""
    w = lib.weight(300, 5120)
    rc = lib.lib.q35mm_matmul_noalloc(w, m, lib.x, lib.y, S)
    rec = lib.take()
    assert rc == 0 and kinds(rec) == ["rows"] * ((m + 7) // 8) and not pointers(rec)


@pytest.mark.parametrize("what", ["matmul", "mlp"])
def test_batch_shares_nothing_with_graphs(lib, what):
    """A graph of a GEMM or a prefill MLP block holds its stream's scratch
    set; row-split matmuls never wrote to it, so the graph could replay
    beside them.  The batch's scratch is none of the graph's."""
    ws = [lib.weight(1664, 5120), lib.weight(1664, 5120), lib.weight(5120, 1664)]
    run = lib.matmul if what == "matmul" else lib.mlp
    arg = ws[0] if what == "matmul" else ws
    assert run(arg, 512, S)[0] == 0
    lib.capture(S)
    rc, rec = run(arg, 512, S)
    held = pointers(rec)
    assert rc == 0 and held
    lib.capture(S, False)
    rc, rec = lib.matmul(ws[0], 63, S)
    assert rc == 0 and "batch" in kinds(rec) and not pointers(rec) & held


def test_batch_does_not_move_the_borrowed_set(lib):
    """A capture on a new stream borrows the set of the last call that has
    one: batches in between, on another stream or captured, change nothing."""
    w = lib.weight(300, 5120)
    assert lib.matmul(w, 1, S)[0] == 0
    lib.capture(S)
    assert lib.matmul(w, 24, S)[0] == 0
    lib.capture(S, False)
    assert lib.matmul(w, 512, T)[0] == 0
    assert lib.matmul(w, 24, U)[0] == 0
    lib.capture(S)
    rc, rec = lib.matmul(w, 512, S)
    assert rc == 0 and "gemm" in kinds(rec)


def test_batch_scratch_is_given_back(lib):
    """q35mm_stream_release frees a stream's batch scratch."""
    w = lib.weight(300, 5120)
    rc, rec = lib.matmul(w, 63, S)
    got = [ln.split()[1] for k, _, ln in rec if k == "malloc"]
    assert rc == 0 and got
    assert lib.lib.q35mm_stream_release(S) == 0
    assert sorted(ln.split()[1] for k, _, ln in lib.take() if k == "free") == sorted(got)


def test_no_memory_runs_eight_at_a_time(lib):
    """Eight tokens need no memory: a batch that gets none runs as they do,
    one that gets less in passes of 32 or 16 tokens, and neither fails."""
    w = lib.weight(30000, 512)
    lib.lib.stub_fail_malloc(1)
    rc, rec = lib.matmul(w, 63, S)
    assert rc == 0 and kinds(rec) == ["rows"] * 8
    lib.lib.stub_fail_malloc(20 << 20)          # 30 MB of range sums at 63 tokens, 15 at 32
    rc, rec = lib.matmul(w, 63, S)
    assert rc == 0 and [f["m"] for k, f, _ in rec if k == "batch"] == ["32", "31"]
    ws = [lib.weight(1664, 512), lib.weight(1664, 512), lib.weight(512, 1664)]
    assert lib.mlp(ws, 1, U)[0] == 0 and lib.mlp(ws, 24, U)[0] == 0
    assert lib.lib.q35mm_stream_release(U) == 0
    assert lib.mlp(ws, 1, U)[0] == 0 and lib.lib.q35mm_mlp(*ws, lib.x, 1e-6, 64, lib.x, U) == 0   # its workspace
    lib.take()
    lib.lib.stub_fail_malloc(1)
    rc, rec = lib.mlp(ws, 24, U)
    assert rc == 0 and kinds(rec) == ["rmsnorm"] + ["pair"] * 3 + ["rows"] * 3


def test_growth_neither_waits_nor_frees(lib):
    """Matmuls of 9..63 tokens never waited for the device; kernels in flight
    may still use the smaller buffer, which stays until the stream's release."""
    w = lib.weight(30000, 512)
    recs = []
    for m in (9, 24, 63, 63):
        rc, rec = lib.matmul(w, m, S)
        assert rc == 0
        recs += rec
    got = [ln.split()[1] for k, _, ln in recs if k == "malloc"]
    assert len(got) >= 2 and not {"device_sync", "free"} & set(kinds(recs))
    assert lib.lib.q35mm_stream_release(S) == 0
    assert sorted(ln.split()[1] for k, _, ln in lib.take() if k == "free") == sorted(got)


def test_beside_another_threads_capture(lib):
    """A capture on another stream does not refuse a first batch: 24 tokens
    on S while T is captured."""
    w = lib.weight(300, 5120)
    lib.capture(T)
    rc, rec = lib.matmul(w, 24, S)
    assert rc == 0 and "batch" in kinds(rec)
    rc, rec = lib.matmul(w, 24, None)           # the null stream cannot be asked
    assert rc == 0 and kinds(rec) == ["rows"] * 3


def test_per_thread_stream_is_not_one_stream(lib):
    """hipStreamPerThread names another stream in each host thread: nothing
    may be kept under that handle."""
    w = lib.weight(300, 5120)
    rc, rec = lib.matmul(w, 24, 2)
    assert rc == 0 and kinds(rec) == ["rows"] * 3


@pytest.mark.parametrize("waves", [4, 8])
def test_mlp_ranges_are_the_paired_kernels(stub_path, monkeypatch, waves):
    """Gate and up of one to eight tokens are summed over four K ranges
    whatever Q35MM_ROWS_WAVES says, down over that many: the batch's too."""
    monkeypatch.setenv("Q35MM_ROWS_WAVES", str(waves))
    lb = Lib(stub_path)
    ws = [lb.weight(1664, 5120), lb.weight(1664, 5120), lb.weight(5120, 1664)]
    seen = {}
    for m in (8, 24):
        rc, rec = lb.mlp(ws, m, S)
        assert rc == 0
        seen[m] = [(k, f["nr"]) for k, f, _ in rec if "nr" in f]
    lb.lib.q35mm_shutdown()
    assert seen[8] == [("pair", "4"), ("rows", str(waves))]
    assert seen[24] == [("batch", "4"), ("batch_swiglu", "4"), ("batch", str(waves))]


@pytest.mark.parametrize("m,cols,rows,batch", [
    (8, 5120, 2048, False), (9, 4096, 48, True), (16, 3968, 1920, False), (9, 3968, 1921, True),
    (9, 3457, 1921, True), (16, 3456, 20000, False), (17, 512, 48, True)])
def test_which_sizes_are_batched(lib, m, cols, rows, batch):
    """From 17 tokens on every row-split weight; 9..16 tokens from 32 K
    blocks on, from 28 on with 16 row groups."""
    rc, rec = lib.matmul(lib.weight(rows, cols), m, S)
    assert rc == 0 and ("batch" in kinds(rec)) == batch


@pytest.mark.parametrize("rows,batch", [((1000, 896), False), ((1000, 1000), True)])
def test_row_groups_of_all_weights_count(lib, rows, batch):
    ws = (C.c_void_p * 2)(*[lib.weight(n, 3584).value for n in rows])
    ys = (C.c_void_p * 2)(lib.y, lib.y)
    assert lib.lib.q35mm_matmul_multi(ws, 2, 9, lib.x, ys, S) == 0
    assert ("batch" in kinds(lib.take())) == batch


def test_scratch_of_all_streams_is_bounded(lib):
    """Streams that come and go without a release: the batch's scratch stays
    within its bound, later streams run eight tokens a launch, and a released
    stream's share serves another."""
    w = lib.weight(60000, 512)               # 62 MB of range sums at 63 tokens
    total = 0
    for i in range(100):
        st = 0x100000 + 16 * i
        rc, rec = lib.matmul(w, 63, st)
        assert rc == 0
        total += sum(int(ln.split()[2]) for k, _, ln in rec if k == "malloc")
        if "batch" in kinds(rec):
            first_without = i + 1
    assert total <= 4 << 30 and 40 < first_without < 100
    rc, rec = lib.matmul(w, 63, 0x100000 + 16 * 99)
    assert rc == 0 and kinds(rec) == ["rows"] * 8
    assert lib.lib.q35mm_stream_release(0x100000) == 0
    rc, rec = lib.matmul(w, 63, 0x100000 + 16 * 99)
    assert rc == 0 and "batch" in kinds(rec)
    for i in range(100):
        assert lib.lib.q35mm_stream_release(0x100000 + 16 * i) == 0
