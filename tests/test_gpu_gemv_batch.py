"""Batched decode (gemv_batch.hip): more than eight tokens of a row-split
weight in one pass over it, below the prefill GEMM.

Its sums are the row-split GEMV's, so every row of a batch is, bit for bit,
the row of a call of one to eight tokens (which the other tests hold against
the oracle): edges of the token tiles (16 and 32), 4..160 K blocks (a last
turn of the four-deep ring of each length), partial blocks both ways, four
and eight K ranges, one row group to hundreds, several weights, values of
any magnitude.  Which calls are batched, and on what scratch, is
test_batch_scratch_cpu.py's.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def _rows_of_small_calls(q, ws, X, gpu):
    import torch
    Ys = [torch.empty((X.shape[0], w.rows), device=gpu) for w in ws]
    for t in range(0, X.shape[0], 8):
        part = [torch.empty((min(8, X.shape[0] - t), w.rows), device=gpu) for w in ws]
        q.matmul_multi(ws, X[t:t + 8].clone(), part)
        for Y, p in zip(Ys, part):
            Y[t:t + 8] = p
    return Ys


def _same_bits(a, b):
    import torch
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


# 9..16 tokens: 32 K blocks or more, or 28 with 16 row groups (fewer go as two small calls)
@pytest.mark.parametrize("m,k,rows", [(9, 3600, (200,)), (16, 4571, (4100,)), (12, 5120, (1300, 48, 5000)),
                                      (10, 20480, (1,)), (17, 5120, (1024,)), (32, 640, (33000,)), (18, 400, (70,)),
                                      (33, 20480, (129,)), (63, 17400, (300,)), (24, 1032, (130, 48, 1, 5000)),
                                      (63, 768, (16300, 70)), (16, 3456, (300,)), (9, 3457, (300,)),
                                      (9, 4200, (200,)), (13, 3457, (2100,)), (16, 3968, (1000, 1000))])
def test_batch_rows_are_small_calls_bitwise(q, wl, gpu, m, k, rows):
    import torch
    ws = [q.Weight(*wl.gen_weight_ragged(k + i, n, k)) for i, n in enumerate(rows)]
    X = torch.from_numpy(wl.gen_act(m, m, k, outlier_frac=0.01)).to(gpu)
    Ys = [torch.empty((m, n), device=gpu) for n in rows]
    q.matmul_multi(ws, X, Ys)
    for Y, R in zip(Ys, _rows_of_small_calls(q, ws, X, gpu)):
        _same_bits(Y, R)
    big = torch.zeros(m * k + 1, device=gpu)   # rows 4 bytes past a 16-byte boundary
    big[1:] = X.reshape(-1)
    Y1 = torch.empty_like(Ys[0])
    q.matmul(ws[0], big[1:].view(m, k), Y1)
    _same_bits(Y1, Ys[0])
    Y2 = torch.empty_like(Ys[0])
    q.matmul_noalloc(ws[0], X, Y2)
    _same_bits(Y2, Ys[0])
    for w in ws:
        w.free()


@pytest.mark.parametrize("m", [16, 40])
def test_batch_wide_values(q, wl, gpu, m):
    """Blocks holding values past 2^96 or infinities are staged shifted."""
    import torch
    k, n = 4200, 300
    w = q.Weight(*wl.gen_weight(5, n, k))
    X = wl.gen_act(6, m, k)
    X[0, 3], X[1, 700], X[2, 999] = np.inf, -np.inf, np.float32(3.4e38)
    X[m - 1, 130], X[5, 131] = np.float32(-2e30), np.nan
    X = torch.from_numpy(X).to(gpu)
    Y = torch.empty((m, n), device=gpu)
    q.matmul(w, X, Y)
    R = _rows_of_small_calls(q, [w], X, gpu)[0]
    assert torch.equal(Y.isnan(), R.isnan())
    _same_bits(Y.nan_to_num(nan=0.0, posinf=np.inf, neginf=-np.inf), R.nan_to_num(nan=0.0, posinf=np.inf, neginf=-np.inf))
    w.free()


@pytest.mark.parametrize("m,H,I", [(9, 3600, 1664), (16, 1032, 4100), (12, 640, 1664), (31, 5120, 1000), (63, 512, 16400)])
def test_batch_mlp_is_small_calls_bitwise(q, wl, gpu, m, H, I):
    """Gate and up in one pass forming silu(gate) * up; residual added."""
    import torch
    w = [q.Weight(*wl.gen_weight(H + i, *s)) for i, s in enumerate(((I, H), (I, H), (H, I)))]
    rng = np.random.default_rng(m)
    nw = torch.from_numpy((rng.standard_normal(H) * 0.1).astype(np.float32)).to(gpu)
    X = torch.from_numpy(rng.standard_normal((m, H)).astype(np.float32)).to(gpu)
    R = X.clone()
    for t in range(0, m, 8):
        part = R[t:t + 8].clone()
        q.mlp(*w, nw, part)
        R[t:t + 8] = part
    q.mlp(*w, nw, X)
    _same_bits(X, R)
    for x in w:
        x.free()


def test_batch_beyond_the_gemm(q, wl, gpu):
    """Block scales too far apart for the prefill GEMM: any m on this path,
    in passes of 64 tokens."""
    import torch
    W, sc = wl.gen_weight(9, 260, 768)
    sc = sc.copy()
    sc[0, 0], sc[0, 1] = 0x6F80, 0x3380     # 2^96 and 2^-24
    w = q.Weight(W, sc)
    X = torch.from_numpy(wl.gen_act(3, 150, 768)).to(gpu)
    Y = torch.empty((150, 260), device=gpu)
    q.matmul(w, X, Y)
    _same_bits(Y, _rows_of_small_calls(q, [w], X, gpu)[0])
    w.free()


def test_batch_capture(q, wl, gpu):
    """Captures run eight tokens a launch, on a stream the library has not
    seen and on one that ran the same call as a batch: both replay to the
    eager bits (test_batch_scratch_cpu.py sees the launches)."""
    import torch
    w = q.Weight(*wl.gen_weight(12, 700, 1024))
    X = torch.from_numpy(wl.gen_act(13, 24, 1024)).to(gpu)
    want = _rows_of_small_calls(q, [w], X, gpu)[0]
    for warm in (False, True):
        s = torch.cuda.Stream()
        Y = torch.zeros((24, 700), device=gpu)
        torch.cuda.synchronize()
        if warm:
            with torch.cuda.stream(s):
                q.matmul(w, X, Y)
            torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            q.matmul(w, X, Y)
        for _ in range(3):
            Y.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            _same_bits(Y, want)
    w.free()


def test_graphs_replayed_at_once(q, wl, gpu):
    """Two graphs of matmuls captured on one stream that has run the same
    calls, replayed on two other streams beside eager calls on the first:
    each gives its own bits."""
    import torch
    w = q.Weight(*wl.gen_weight(14, 5120, 5120))
    Xs = [torch.from_numpy(wl.gen_act(15 + i, 40, 5120)).to(gpu) for i in range(3)]
    want = [_rows_of_small_calls(q, [w], X, gpu)[0] for X in Xs]
    Ys = [torch.zeros((40, 5120), device=gpu) for _ in range(3)]
    s, other = torch.cuda.Stream(), [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        q.matmul(w, Xs[2], Ys[2])
    torch.cuda.synchronize()
    gs = []
    for X, Y in zip(Xs[:2], Ys):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            q.matmul(w, X, Y)
        gs.append(g)
    for _ in range(3):
        for Y in Ys:
            Y.zero_()
        torch.cuda.synchronize()
        for _ in range(10):
            for g, o in zip(gs, other):
                with torch.cuda.stream(o):
                    g.replay()
            with torch.cuda.stream(s):
                q.matmul(w, Xs[2], Ys[2])
        torch.cuda.synchronize()
        for Y, R in zip(Ys, want):
            _same_bits(Y, R)
    q.stream_release(s.cuda_stream)
    w.free()


def test_eight_ranges_keep_the_bits():
    """Q35MM_ROWS_WAVES=8 (read when the library starts, so in a process of
    its own): the batch sums eight K ranges as one to eight tokens do, the
    MLP block's gate and up four."""
    code = r"""
import sys, numpy as np, torch
sys.path.insert(0, %r)
import q35mm as q, workload as wl
gpu = torch.device("cuda:0")
def same(a, b):
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
for m, k, n in ((9, 4200, 200), (24, 1032, 300), (63, 5120, 129)):
    print("matmul", m, k, n, flush=True)
    w = q.Weight(*wl.gen_weight(k, n, k))
    X = torch.from_numpy(wl.gen_act(m, m, k)).to(gpu)
    Y, R = torch.empty((m, n), device=gpu), torch.empty((m, n), device=gpu)
    q.matmul(w, X, Y)
    for t in range(m):
        q.matmul(w, X[t:t + 1], R[t:t + 1])
    same(Y, R)
for m, H, I in ((17, 2048, 1664), (40, 1032, 1100)):
    print("mlp", m, H, I, flush=True)
    ws = [q.Weight(*wl.gen_weight(H + i, *s)) for i, s in enumerate(((I, H), (I, H), (H, I)))]
    nw = torch.zeros(H, device=gpu)
    X = torch.from_numpy(wl.gen_act(m, m, H)).to(gpu)
    R = X.clone()
    for t in range(0, m, 8):
        part = R[t:t + 8].clone()
        q.mlp(*ws, nw, part)
        R[t:t + 8] = part
    q.mlp(*ws, nw, X)
    same(X, R)
print("done")
""" % os.path.join(ROOT, "qwen38-in-c_amd")
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, Q35MM_ROWS_WAVES="8"),
                         capture_output=True, text=True, timeout=110)
    print(out.stdout, flush=True)
    assert out.returncode == 0 and out.stdout.rstrip().endswith("done"), out.stdout + out.stderr[-2000:]


@pytest.mark.parametrize("m", [16, 40])
def test_wide_values_leave_other_tokens_alone(q, wl, gpu, m):
    """A wide value shifts its K block for the tokens one launch of the
    row-split GEMV takes with it (its eight), whose values below 2^-62 lose
    bits; the rest of its tile keeps theirs."""
    import torch
    k, n = 4200, 300
    w = q.Weight(*wl.gen_weight(7, n, k))
    rng = np.random.default_rng(m)
    X = rng.standard_normal((m, k)).astype(np.float32)
    X[:, 128:256] *= np.float32(2.0 ** -70)      # whole blocks of tiny values
    X[:, 3456:] *= np.float32(2.0 ** -80)        # the last, partial block too
    X[0, 130], X[m - 1, 3500] = np.float32(2e30), np.float32(-3e29)
    X = torch.from_numpy(X).to(gpu)
    X[1:m - 1, :128], X[1:m - 1, 256:3456] = 0.0, 0.0    # nothing else hides them
    Y = torch.empty((m, n), device=gpu)
    q.matmul(w, X, Y)
    _same_bits(Y, _rows_of_small_calls(q, [w], X, gpu)[0])
    w.free()


def test_wide_products_in_the_mlp(q, wl, gpu):
    """The same for silu(gate) * up: token 0's products are near 1e30 (column
    0 of x reaches the norm weight 1e18), the others' near 1e-20, beside a
    residual of 1e-18."""
    import torch
    m, H, I = 24, 1024, 1664
    w = []
    for i, (n, k) in enumerate(((I, H), (I, H), (H, I))):
        W, sc = wl.gen_weight(90 + i, n, k)
        w.append(q.Weight(W, sc - np.uint16(8 << 7) if i < 2 else sc))   # gate and up times 2^-8
    nw = np.full(H, -1.0 + 2.0 ** -24, np.float32)
    nw[0] = 1e18
    x = np.random.default_rng(3).standard_normal((m, H)).astype(np.float32) * np.float32(1e-18)
    x[1:, 0], x[0, 0] = 0.0, 5e-18
    nw, X = torch.from_numpy(nw).to(gpu), torch.from_numpy(x).to(gpu)
    R, X0 = X.clone(), X.clone()
    for t in range(0, m, 8):
        part = R[t:t + 8].clone()
        q.mlp(*w, nw, part, 0.0)
        R[t:t + 8] = part
    q.mlp(*w, nw, X, 0.0)
    assert torch.isfinite(R).all() and (R[0].abs().max() > 1e26) and not torch.equal(R[8:], X0[8:])
    _same_bits(X, R)
    for v in w:
        v.free()


def test_first_batch_beside_a_capture(q, wl, gpu):
    """A batch whose scratch is allocated while another stream is captured:
    the call works and the capture stays valid."""
    import torch
    w = q.Weight(*wl.gen_weight(16, 700, 5120))
    X = torch.from_numpy(wl.gen_act(17, 24, 5120)).to(gpu)
    want = _rows_of_small_calls(q, [w], X, gpu)[0]
    Y, Z = torch.zeros_like(want), torch.zeros_like(want)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    q.stream_release(t.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        q.matmul(w, X, Y)
        q.matmul(w, X, Z, stream=t.cuda_stream)
    torch.cuda.synchronize()
    _same_bits(Z, want)
    for _ in range(3):
        Y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        _same_bits(Y, want)
    w.free()
