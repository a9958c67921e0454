"""Workloads of the FP8 block-dequant matmul library, as a model's program runs them.

Each case is one pass through the public entry points (qwen38-in-c_amd/q35mm.py
over libq35mm.so): single projections, multi-weight projections, the MLP
block, a whole layer's matmul path, the BF16 lm_head and the host-pointer
drop-in call.  Sizes are the model's projections (workload.py) and the
benchmark's; tokens run from one (decode) over batches of 2..63 (batched
decode, short prompts) to prefills of 64..2048.

Weights are N(0, 0.02^2) fp32 quantized per 128x128 block (scale = amax/448 in
bf16, codes nearest e4m3); "ragged" weights draw each block's amax
log-uniform in [1e-4, 1e2].  Activations are N(0, 1) fp32 with a few outlier
channels, as hidden states have.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "qwen38-in-c_amd")   # the working folder is the repository's root
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import q35mm  # noqa: E402

DEV = "cuda:0"
EPS = 1e-6
HIDDEN, INTER, VOCAB = 5120, 17408, 248320
DELTANET_IN = (10240, 6144, 48, 48)      # in_proj_qkv, in_proj_z, in_proj_a, in_proj_b
GQA_IN = (12288, 1024, 1024)             # q, k, v
GEMM_MIN_M = 64                          # tokens from which the bf16 prefill GEMM runs
MAX_TOKENS = 2048
MAX_WEIGHT = 400 << 20                   # bytes of FP8 weights in one drawn case


def listed():
    return [
        # the smallest call of a decode step: one GQA k projection, one token
        _matmul("k_proj_m1", 1, 5120, 1024),
        # the drop-in C ABI as the reference's engine calls it: host pointers, one token
        _case("host_5120_m1", "host", 1, 5120, (5120,)),
        # one token through all matmuls of a Gated DeltaNet layer: in_proj (four weights, one call), out_proj, MLP block
        _layer("layer_m1", 1),
        # eight sequences decoded together
        _layer("layer_m8", 8),
        # two dozen sequences decoded together
        _layer("layer_m24", 24),
        # ragged shape with extreme block scales and outlier activations: partial blocks in both directions
        _case("ragged_m37", "matmul", 37, 4736, (3000,), ragged=True),
        # a short prompt through a GQA layer's q, k, v
        _case("gqa_qkv_m61", "multi", 61, 5120, GQA_IN),
        # a prompt of a hundred tokens through the MLP block
        _case("mlp_m100", "mlp", 100, HIDDEN, (INTER,)),
        # prefill, one projection alone (out_proj of the straggler path)
        _matmul("out_proj_m512", 512, 6144, 5120),
        # prefill of 512 tokens through all matmuls of a layer
        _layer("layer_m512", 512),
        # a long prompt through the MLP block: the largest
        _case("mlp_m2048", "mlp", 2048, HIDDEN, (INTER,)),
        # the BF16 lm_head of one token
        _case("lm_head", "bf16", 1, HIDDEN, (VOCAB,)),
    ]


def _case(name, kind, m, k, rows, ragged=False):
    c = {"kind": kind, "m": m, "k": k, "ragged": ragged}
    for i in range(4):
        c["rows%d" % i] = rows[i] if i < len(rows) else 0
    if name:
        c["name"] = name
    return c


def _matmul(name, m, k, n):
    return _case(name, "matmul", m, k, (n,))


def _layer(name, m):
    return _case(name, "layer", m, HIDDEN, DELTANET_IN)


def _rows(case):
    return [case["rows%d" % i] for i in range(4) if case["rows%d" % i]]


def draw(rng):
    """A case of the listed ranges: every kind, sizes log-uniform, multiples of 128, of 8 and odd ones."""

    def size(lo, hi):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        step = rng.choice((128, 128, 8, 1))
        return max(lo, min(hi, v // step * step))

    kind = rng.choice(("matmul", "matmul", "multi", "mlp", "layer", "bf16", "host"))
    m = max(1, min(MAX_TOKENS, int(round(math.exp(rng.uniform(0.0, math.log(MAX_TOKENS)))))))
    if kind == "layer":
        return _layer(None, min(m, 1024))
    if kind == "bf16":
        return _case(None, "bf16", 1, size(1024, 6144), (size(32000, 200000),))
    if kind == "host":
        return _case(None, "host", min(m, 512), size(1024, 8192), (size(1024, 8192),))
    if kind == "mlp":
        h = size(1024, 6144)
        return _case(None, "mlp", m, h, (min(size(2048, 20000), MAX_WEIGHT // (3 * h)),))
    k = size(1024, 17408)
    n = rng.choice((1, 2, 3, 4)) if kind == "multi" else 1
    rows = tuple(min(size(48, 20000), MAX_WEIGHT // (n * k)) for _ in range(n))
    return _case(None, kind, m, k, rows, ragged=kind == "matmul" and rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt * 7919) & 0x7FFFFFFFFFFF)
    return g


def _weight(seed, salt, n, k, ragged=False):
    """(codes uint8 [n][k], bf16 scale bits int16 [NB][KB]) on the device."""
    g = _gen(seed, salt)
    nb, kb = (n + 127) // 128, (k + 127) // 128
    w = torch.empty((n, k), device=DEV).normal_(0.0, 0.02, generator=g)
    pad = torch.zeros((nb * 128, kb * 128), device=DEV)
    pad[:n, :k] = w
    blk = pad.view(nb, 128, kb, 128)
    amax = blk.abs().amax(dim=(1, 3))
    if ragged:
        want = torch.pow(10.0, torch.empty((nb, kb), device=DEV).uniform_(-4.0, 2.0, generator=g))
        blk.mul_((want / amax)[:, None, :, None])
        amax = want
    sc = (amax / 448.0).to(torch.bfloat16)
    codes = (blk / sc.float()[:, None, :, None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    codes = codes.view(torch.uint8).reshape(nb * 128, kb * 128)[:n, :k].contiguous()
    return codes, sc.view(torch.int16)


def _act(seed, salt, m, k, outliers=4):
    g = _gen(seed, salt)
    x = torch.empty((m, k), device=DEV).normal_(generator=g)
    ch = torch.randint(0, k, (outliers,), device=DEV, generator=g)
    x[:, ch] *= 20.0
    return x


def _ragged_act(seed, salt, m, k):
    g = _gen(seed, salt)
    x = torch.empty((m, k), device=DEV).normal_(generator=g)
    hit = torch.empty((m, k), device=DEV).uniform_(generator=g) < 0.01
    return torch.where(hit, x * 100.0, x)


def _norm_weight(seed, salt, n):
    return torch.empty(n, device=DEV).normal_(0.0, 0.1, generator=_gen(seed, salt))


def _resident(seed, salt, n, k, ragged=False):
    codes, sc = _weight(seed, salt, n, k, ragged)
    return q35mm.Weight(codes.cpu().numpy(), sc.cpu().numpy().view(np.uint16))


def _bf16_weight(seed, n, k):
    return torch.empty((n, k), device=DEV, dtype=torch.bfloat16).normal_(0.0, 0.02, generator=_gen(seed, 1))


def _input(case, seed):
    m, k = case["m"], case["k"]
    return _ragged_act(seed, 2, m, k) if case["ragged"] else _act(seed, 2, m, k)


# Salts of a layer's or MLP's tensors.
_S_IN, _S_OUT, _S_GATE, _S_UP, _S_DOWN, _S_NORM, _S_ATT, _S_RES = 10, 20, 21, 22, 23, 24, 25, 26


def prepare(case, seed):
    kind, m, k, rows = case["kind"], case["m"], case["k"], _rows(case)
    st = {"kind": kind}
    if kind == "bf16":
        st["w"] = _bf16_weight(seed, rows[0], k)
        st["x"] = _act(seed, 2, 1, k).reshape(k)
        st["y"] = torch.empty(rows[0], device=DEV)
        return st
    if kind == "host":
        codes, sc = _weight(seed, _S_IN, rows[0], k)
        st["W"], st["sc"] = codes.cpu().numpy(), sc.cpu().numpy().view(np.uint16)
        st["X"] = _input(case, seed).cpu().numpy()
        q35mm.mm_fp8_batch(st["W"], st["sc"], np.zeros((1, k), np.float32))   # bound once, resident from then on
        return st
    if kind in ("matmul", "multi", "layer"):
        st["x"] = _input(case, seed)
        st["w"] = [_resident(seed, _S_IN + i, n, k, case["ragged"]) for i, n in enumerate(rows)]
        st["y"] = [torch.empty((m, n), device=DEV) for n in rows]
    if kind == "layer":
        st["att"] = _act(seed, _S_ATT, m, 6144)
        st["w_out"] = _resident(seed, _S_OUT, HIDDEN, 6144)
        st["proj"] = torch.empty((m, HIDDEN), device=DEV)
    if kind in ("mlp", "layer"):
        inter = rows[0] if kind == "mlp" else INTER
        st["gate"] = _resident(seed, _S_GATE, inter, k)
        st["up"] = _resident(seed, _S_UP, inter, k)
        st["down"] = _resident(seed, _S_DOWN, k, inter)
        st["norm"] = _norm_weight(seed, _S_NORM, k)
        st["res"] = _act(seed, _S_RES, m, k)
        st["h"] = torch.empty((m, k), device=DEV)
        if kind == "mlp":
            st["proj"] = _act(seed, _S_ATT, m, k, outliers=0)
    return st


def run(state):
    s, kind = state, state["kind"]
    if kind == "bf16":
        q35mm.bf16_gemv(s["w"], s["x"], s["y"])
        return s["y"]
    if kind == "host":
        return q35mm.mm_fp8_batch(s["W"], s["sc"], s["X"])
    if kind == "matmul":
        q35mm.matmul(s["w"][0], s["x"], s["y"][0])
        return s["y"][0]
    outs = []
    if kind in ("multi", "layer"):
        q35mm.matmul_multi(s["w"], s["x"], s["y"])
        outs += s["y"]
    if kind == "layer":
        q35mm.matmul(s["w_out"], s["att"], s["proj"])
        outs.append(s["proj"])
    if kind in ("mlp", "layer"):
        torch.add(s["res"], s["proj"], out=s["h"])   # the attention's residual add
        q35mm.mlp(s["gate"], s["up"], s["down"], s["norm"], s["h"], EPS)
        outs.append(s["h"])
    return outs


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _mm_work(m, k, n):
    nb, kb = (n + 127) // 128, (k + 127) // 128
    return n * k + 4 * nb * kb + 4 * m * n, 2 * m * n * k


def work(case):
    kind, m, k, rows = case["kind"], case["m"], case["k"], _rows(case)
    if kind == "bf16":
        return {"bytes": 2 * rows[0] * k + 4 * (k + rows[0]), "flops": 2 * rows[0] * k}
    b = f = 0
    if kind != "mlp":
        b += 4 * m * k
        for n in rows:
            wb, wf = _mm_work(m, k, n)
            b, f = b + wb, f + wf
    if kind == "layer":
        wb, wf = _mm_work(m, 6144, HIDDEN)
        b, f = b + wb + 4 * m * 6144, f + wf
    if kind in ("mlp", "layer"):
        inter = rows[0] if kind == "mlp" else INTER
        for n, kk in ((inter, k), (inter, k), (k, inter)):
            nb, kb = (n + 127) // 128, (kk + 127) // 128
            b, f = b + n * kk + 4 * nb * kb, f + 2 * m * n * kk
        b += 3 * 4 * m * k + 4 * k      # residual and attention output in, residual stream out
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Below GEMM_MIN_M tokens activations stay fp32 and sums are fp32: outputs measure 1e-7 to 2.5e-7 from 64
    bits (the BF16 matvec's sequential fp32 chains 4.5e-7).  From there on activations are rounded to bf16: 1.7e-3
    for one product, 2.7e-3 to 3.1e-3 for the MLP block, whose products are rounded twice."""
    if case["kind"] == "bf16":
        return {"rel": 2e-6, "max": 1e-4}
    if case["m"] < GEMM_MIN_M:
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _dequant64(seed, salt, n, k, ragged=False):
    codes, sc = _weight(seed, salt, n, k, ragged)
    s = sc.view(torch.bfloat16).double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    return codes.view(torch.float8_e4m3fn).float().double() * s


def _mm64(x, seed, salt, n, k, ragged=False):
    return x.double() @ _dequant64(seed, salt, n, k, ragged).t().contiguous()


def exact(case, seed):
    kind, m, k, rows = case["kind"], case["m"], case["k"], _rows(case)
    if kind == "bf16":
        w, x = _bf16_weight(seed, rows[0], k), _act(seed, 2, 1, k).reshape(k).double()
        return torch.cat([w[i:i + 8192].double() @ x for i in range(0, rows[0], 8192)])
    if kind == "host":
        return _mm64(_input(case, seed), seed, _S_IN, rows[0], k).cpu().numpy()
    outs = []
    if kind in ("matmul", "multi", "layer"):
        x = _input(case, seed)
        outs = [_mm64(x, seed, _S_IN + i, n, k, case["ragged"]) for i, n in enumerate(rows)]
        if kind == "matmul":
            return outs[0]
    if kind == "layer":
        proj = _mm64(_act(seed, _S_ATT, m, 6144), seed, _S_OUT, HIDDEN, 6144)
        outs.append(proj)
    if kind in ("mlp", "layer"):
        inter = rows[0] if kind == "mlp" else INTER
        if kind == "mlp":
            proj = _act(seed, _S_ATT, m, k, outliers=0).double()
        h = _act(seed, _S_RES, m, k).double() + proj
        inv = torch.rsqrt(h.square().mean(dim=1, keepdim=True) + EPS)
        xn = h * inv * (1.0 + _norm_weight(seed, _S_NORM, k).double())
        g, u = _mm64(xn, seed, _S_GATE, inter, k), _mm64(xn, seed, _S_UP, inter, k)
        outs.append(h + _mm64(torch.nn.functional.silu(g) * u, seed, _S_DOWN, k, inter))
    return outs
