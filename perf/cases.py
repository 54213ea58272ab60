"""Measured workloads of the MoE decode path: what a program that serves a
qwen3moe model with this library has it do, from one small matrix-vector
product to whole prompts and generations of an engine model.

Six kinds of case:

  matvec     one dense projection (styx_op_matvec): attention q/k/v/o
             matrices at the small end, the LM head at the large end
  ffn        the half of a decode layer after attention, op by op
             (styx_op_matvec o-proj, styx_op_router_topk,
             styx_op_moe_gate_up, styx_op_moe_down_reduce)
  attn       paged decode attention of one layer (styx_op_attn_decode)
  pipelines  one whole decode layer recorded in a command batch with the
             reference engine's own pipelines (rms_norm, mul_mat_vec,
             rope, attn_decode, ...), weights in GGUF layout
  split      an expert tensor's conversion from GGUF to the split layout,
             the device work of loading a model
  model      a GGUF model in the engine: prompt, greedy generation and the
             logits after it; all experts in HBM or half of them in pinned
             host memory

Shapes are those of the 30B-A3B, 235B-A22B and 80B-A3B configurations that
bench.py and the tests use, and generic sizes around them.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import struct
import tempfile
import zlib

import numpy as np
import torch

from styx_amd import _lib as L
from styx_amd import gguf_io
from styx_amd.model import MoeModel
from styx_amd.runtime import Batch, Gpu, Kernel

Q8_0, Q4_K, Q5_K, Q6_K = L.Q8_0, L.Q4_K, L.Q5_K, L.Q6_K
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
EPS = 1e-6
ROPE_BASE = 1e6
SIGMA = 0.02
DEV = "cuda"


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # the k projection of a 30B-A3B layer with its RMSNorm: the smallest
        # call a decode step makes
        dict(name="matvec_k_proj", kind="matvec", type="q8_0", rows=512, cols=2048, norm=True),
        # the LM head of the 30B-A3B shape, q6_K as GGUF files usually hold it
        dict(name="matvec_lm_head", kind="matvec", type="q6_k", rows=151936, cols=2048, norm=True),
        # after attention, 30B-A3B layer with the mixed K-quant experts
        dict(name="ffn_30b", kind="ffn", H=2048, F=768, E=128, k=8, qd=4096, attn_type="q8_0",
             gate="q4_k", up="q5_k", down="q6_k"),
        # after attention, 235B-A22B layer with q4_K experts
        dict(name="ffn_235b", kind="ffn", H=4096, F=1536, E=128, k=8, qd=8192, attn_type="q8_0",
             gate="q4_k", up="q4_k", down="q4_k"),
        # attention of a 30B-A3B layer in a conversation of about a thousand tokens
        dict(name="attn_1k", kind="attn", heads=32, kv=4, hd=128, context=1021, norms=True),
        # attention of a 235B-A22B layer at the longest context served
        dict(name="attn_32k", kind="attn", heads=64, kv=4, hd=128, context=32768, norms=True),
        # a 30B-A3B layer through the reference's pipelines early in a
        # generation, q8_0 throughout
        dict(name="pipelines_q8_short", kind="pipelines", H=2048, heads=32, kv=4, hd=128, E=128,
             k=8, F=768, attn_type="q8_0", gate="q8_0", up="q8_0", down="q8_0", context=145),
        # the same layer with K-quant experts at the reference's full context
        dict(name="pipelines_k_4k", kind="pipelines", H=2048, heads=32, kv=4, hd=128, E=128, k=8,
             F=768, attn_type="q8_0", gate="q4_k", up="q5_k", down="q6_k", context=4000),
        # one gate tensor of a 30B-A3B layer on its way into HBM
        dict(name="split_q4k_experts", kind="split", type="q4_k", rows=768, cols=2048, experts=128),
        # reading a prompt of a few hundred tokens, then the first new ones
        dict(name="model_prompt_384", kind="model", layers=2, H=2048, heads=32, kv=4, hd=128,
             E=128, k=8, F=768, shexp=False, vocab=32768, attn_type="q8_0", mix=True,
             prompt=384, new=2, host=False),
        # a short question and an answer: decode dominates
        dict(name="model_answer_48", kind="model", layers=2, H=2048, heads=32, kv=4, hd=128,
             E=128, k=8, F=768, shexp=False, vocab=32768, attn_type="q8_0", mix=True,
             prompt=17, new=48, host=False),
        # a model larger than its HBM budget: half of the experts, the less
        # popular, stay in pinned host memory
        dict(name="model_offload_96", kind="model", layers=2, H=2048, heads=32, kv=4, hd=128,
             E=128, k=8, F=768, shexp=False, vocab=32768, attn_type="q8_0", mix=True,
             prompt=96, new=8, host=True),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "ffn", "attn", "pipelines", "split", "model"])
    kq = ["q4_k", "q5_k", "q6_k"]
    if kind == "matvec":
        t = rng.choice(list(TYPES))
        cols = 256 * rng.choice([3, 4, 6, 8, 12, 16, 24, 32]) if t == "q8_0" else \
            512 * rng.choice([1, 2, 3, 4, 6, 8, 16])
        rows = _logint(rng, 200, min(151936, 151936 * 2048 // cols))
        if t == "q5_k":  # the split layout takes q5_K blocks in groups of 8
            g = 8 // math.gcd(8, cols // 256)
            rows = -(-rows // g) * g
        return dict(kind=kind, type=t, rows=rows, cols=cols, norm=rng.random() < 0.5)
    if kind == "split":
        t = rng.choice(list(TYPES))
        return dict(kind=kind, type=t, rows=8 * _logint(rng, 8, 96), cols=256 * rng.randint(1, 8),
                    experts=_logint(rng, 1, 128))
    if kind == "attn":
        kv = rng.choice([1, 2, 4, 8])
        gqa = rng.choice([1, 2, 4, 8, 16])
        hd = rng.choice([64, 128, 128, 256])
        return dict(kind=kind, heads=kv * gqa, kv=kv, hd=hd,
                    context=_logint(rng, 1, 32768 * 512 // (kv * hd) if kv * hd > 512 else 32768),
                    norms=rng.random() < 0.8)
    H = 256 * rng.choice([4, 6, 8])
    F = 256 * rng.choice([1, 2, 3, 4])
    E = rng.choice([32, 64, 128])
    k = rng.choice([4, 6, 8, 10])
    if rng.random() < 0.3:
        gate = up = down = "q8_0"
    else:
        gate, up, down = (rng.choice(kq) for _ in range(3))
    if kind == "ffn":
        return dict(kind=kind, H=H, F=F, E=E, k=k, qd=2048 * rng.choice([1, 2]),
                    attn_type=rng.choice(["q8_0", "q6_k"]), gate=gate, up=up, down=down)
    kv = rng.choice([2, 4])
    heads = kv * rng.choice([4, 8])
    if kind == "pipelines":
        return dict(kind=kind, H=H, heads=heads, kv=kv, hd=rng.choice([64, 128]), E=E, k=k, F=F,
                    attn_type=rng.choice(["q8_0", "q4_k"]), gate=gate, up=up, down=down,
                    context=_logint(rng, 1, 4000))
    host = rng.random() < 0.3
    return dict(kind="model", layers=2, H=H, heads=heads, kv=kv, hd=128, E=E, k=k, F=min(F, 768),
                shexp=rng.random() < 0.3, vocab=8192, attn_type=rng.choice(["q8_0", "q6_k"]),
                mix=rng.random() < 0.7, prompt=_logint(rng, 1, 96 if host else 384),
                new=_logint(rng, 1, 8 if host else 24), host=host)


# ----------------------------------------------------------- seeded values --
def _gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed(((int(seed) & 0xFFFFFFFF) << 32) ^ zlib.crc32(name.encode()))
    return g


def _normal(seed, name, *shape, scale=1.0, mean=0.0):
    return torch.randn(*shape, generator=_gen(seed, name), device=DEV) * scale + mean


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


def _quant(seed, name, t, n):
    """n zero-mean weights of spread about SIGMA as GGUF blocks of type t."""
    el, by = L.BLOCK[t]
    nb = n // el
    g = _gen(seed, name)

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, (nb, *shape), generator=g, device=DEV, dtype=torch.uint8)

    vary = 0.75 + 0.5 * torch.rand(nb, generator=g, device=DEV)
    out = torch.empty(nb, by, dtype=torch.uint8, device=DEV)
    if t == Q8_0:
        out[:, 0:2] = _f16_bytes(SIGMA / 73.6 * vary)
        out[:, 2:] = ints(0, 255, 32) - 127  # int8 values of [-127, 127]
        return out
    if t == Q6_K:
        out[:, 0:192] = ints(0, 256, 192)
        sign = ints(0, 2, 16)
        sc = ints(32, 128, 16)
        out[:, 192:208] = torch.where(sign > 0, sc, (0 - sc))
        out[:, 208:210] = _f16_bytes(SIGMA / (18.5 * 83.0) * vary)
        return out
    mid, rms = (7.5, 4.61) if t == Q4_K else (15.5, 9.23)
    d = SIGMA / (rms * 48.4) * vary
    out[:, 0:2] = _f16_bytes(d)
    out[:, 2:4] = _f16_bytes(mid * d)
    s = ints(32, 64, 8)  # scales and minima alike: weights d s (q - mid)
    out[:, 4:8] = s[:, :4] | ((s[:, 4:] >> 4) << 6)
    out[:, 8:12] = out[:, 4:8]
    out[:, 12:16] = (s[:, 4:] & 15) | ((s[:, 4:] & 15) << 4)
    out[:, 16:] = ints(0, 256, by - 16)
    return out


def _f64(b2):
    return b2.contiguous().view(torch.float16).to(torch.float64)


def _dequant64(t, b):
    """GGUF blocks [nb, bytes] to [nb, elements] in 64 bits."""
    nb = b.shape[0]
    if t == Q8_0:
        return b[:, 2:].contiguous().view(torch.int8).to(torch.float64) * _f64(b[:, 0:2])
    if t == Q6_K:
        d = _f64(b[:, 208:210])
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64) * d  # [nb, 16]
        ql = b[:, 0:128].view(nb, 2, 2, 32)   # [half, run, 32]
        qh = b[:, 128:192].view(nb, 2, 1, 32)
        lo = torch.stack([ql[:, :, 0], ql[:, :, 1], ql[:, :, 0], ql[:, :, 1]], 2)
        sh = torch.tensor([0, 0, 4, 4], device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        hs = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = ((lo >> sh) & 15) | (((qh >> hs) & 3) << 4)  # [nb, 2, 4, 32]
        q = q.to(torch.float64) - 32.0
        return (q.view(nb, 16, 16) * sc.view(nb, 16, 1)).view(nb, 256)
    d, dmin = _f64(b[:, 0:2]), _f64(b[:, 2:4])
    s, m, hi = b[:, 4:8], b[:, 8:12], b[:, 12:16]
    sc = torch.cat([s & 63, (hi & 15) | ((s >> 6) << 4)], 1).to(torch.float64) * d
    mn = torch.cat([m & 63, (hi >> 4) | ((m >> 6) << 4)], 1).to(torch.float64) * dmin
    qs = b[:, 16:144] if t == Q4_K else b[:, 48:176]
    qs = qs.reshape(nb, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32)
    if t == Q5_K:
        sh = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
        q = q | (((b[:, 16:48].view(nb, 1, 32) >> sh) & 1) << 4)
    return (q.to(torch.float64) * sc.view(nb, 8, 1) - mn.view(nb, 8, 1)).view(nb, 256)


def _mul64(t, blocks, rows, cols, x):
    """x [n, cols] times the transposed rows x cols matrix, in 64 bits."""
    per = cols // L.BLOCK[t][0]
    step = max(1, (1 << 25) // cols)
    outs = []
    for r in range(0, rows, step):
        n = min(step, rows - r)
        w = _dequant64(t, blocks[r * per:(r + n) * per]).view(n, cols)
        outs.append(x @ w.T)
    return torch.cat(outs, 1)


def _rms64(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rope64(x, pos, hd):
    """x [n, heads, hd] rotated (NEOX pairs) at positions pos [n]."""
    half = hd // 2
    inv = torch.tensor([ROPE_BASE ** (-2.0 * i / hd) for i in range(half)], dtype=torch.float64,
                       device=x.device)
    th = pos.double()[:, None] * inv[None]
    c, s = th.cos()[:, None], th.sin()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend64(q, k, v, pos):
    """q [n, heads, hd] at positions pos over k/v [t, kv, hd], causal."""
    n, heads, hd = q.shape
    t, kv, _ = k.shape
    out = torch.empty_like(q)
    seen = torch.arange(t, device=q.device)[None] <= pos[:, None]
    for h in range(kv):
        g = heads // kv
        s = torch.einsum("ngd,td->ngt", q[:, h * g:(h + 1) * g], k[:, h].contiguous())
        s = s / math.sqrt(hd)
        s = s.masked_fill(~seen[:, None], -math.inf)
        out[:, h * g:(h + 1) * g] = torch.softmax(s, -1) @ v[:, h].contiguous()
    return out


def _moe64(x, logits, k, gate, up, down, H, F):
    """Routed experts of normalised x [n, H]: sum of the k best by softmax
    weight, renormalised; gate/up/down are (type, blocks)."""
    p = torch.softmax(logits, -1)
    w, e = torch.topk(p, k, -1)
    w = w / w.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for ex in e.unique().tolist():
        tok, slot = (e == ex).nonzero(as_tuple=True)
        out[tok] += _swiglu64(x[tok], ex, gate, up, down, H, F) * w[tok, slot][:, None]
    return out, w, e


def _swiglu64(x, ex, gate, up, down, H, F):
    def one(tb, rows, cols, v):
        t, b = tb
        per = rows * cols // L.BLOCK[t][0]
        return _mul64(t, b[ex * per:(ex + 1) * per], rows, cols, v)
    g, u = one(gate, F, H, x), one(up, F, H, x)
    return one(down, H, F, g * torch.sigmoid(g) * u)


# ------------------------------------------------------------------- state --
_GPU = None


def _gpu():
    """The process's device handle, opened once, as a program holds it."""
    global _GPU
    if _GPU is None:
        _GPU = Gpu(0)
    return _GPU


class State:
    """What a program keeps between calls; frees the library's objects."""

    def __init__(self, case):
        self.case, self.gpu, self.owned = case, _gpu(), []

    def own(self, o, close="free"):
        self.owned.append((o, close))
        return o

    def __del__(self):
        for o, close in reversed(self.owned):
            getattr(o, close)()


class _Ptr:
    def __init__(self, buf, shape, typestr):
        self.buf = buf  # a Buffer frees its memory with its last reference
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, version=2,
                                             data=(buf.ptr, False), strides=None)


def _view(buf, dtype, *shape):
    """A library buffer as a torch tensor."""
    ts = {torch.float32: "<f4", torch.uint8: "|u1", torch.int32: "<i4"}[dtype]
    return torch.as_tensor(_Ptr(buf, shape, ts), device=DEV)


def _split(s, t, blocks, rows, cols, nmat=1):
    """Split-layout copy of GGUF blocks, as a program lays weights out once."""
    out = torch.empty(blocks.numel(), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    L.check(s.gpu.lib.styx_op_to_split(s.gpu.h, t, blocks.data_ptr(), out.data_ptr(),
                                       rows * cols // L.BLOCK[t][0], nmat))
    s.gpu.sync()
    return out


def _rope_table(hd, n):
    out = np.empty((n, hd // 2, 2), np.float64)
    _gpu().lib.styx_rope_table(C.c_float(ROPE_BASE), hd, n, out.ctypes.data)
    return torch.from_numpy(out).to(DEV)


def _norm_w(seed, name, n):
    return _normal(seed, name, n, scale=0.1, mean=1.0)


def prepare(case, seed):
    s = State(case)
    globals()["_prepare_" + case["kind"]](s, case, seed)
    torch.cuda.synchronize()
    return s


def run(s):
    return globals()["_run_" + s.case["kind"]](s)


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def work(case):
    b, f = globals()["_work_" + case["kind"]](case)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # sums of f32 products in another order (and 23-bit activation limbs)
    # differ by a few 1e-7 of the result's norm; a layer or a model carries
    # such differences on through norms, softmax and SiLU
    return {"matvec": {"rel": 1e-6, "max": 1e-5},
            "ffn": {"rel": 1e-6, "max": 1e-5},
            "attn": {"rel": 1e-6, "max": 1e-5},
            "pipelines": {"rel": 1e-6, "max": 1e-5},
            "split": "exact",
            "model": {"rel": 2e-6, "max": 2e-5, "differ": 0.0}}[case["kind"]]


def _mat_bytes(t, n):
    el, by = L.BLOCK[TYPES[t]]
    return n // el * by


# ------------------------------------------------------------------ matvec --
def _matvec_inputs(case, seed):
    rows, cols, t = case["rows"], case["cols"], TYPES[case["type"]]
    return (_quant(seed, "w", t, rows * cols), _normal(seed, "x", cols, scale=1.5),
            _norm_w(seed, "norm", cols))


def _prepare_matvec(s, case, seed):
    blocks, s.x, s.nw = _matvec_inputs(case, seed)
    s.w = _split(s, TYPES[case["type"]], blocks, case["rows"], case["cols"])
    s.y = torch.empty(case["rows"], device=DEV)


def _run_matvec(s):
    c = s.case
    L.check(s.gpu.lib.styx_op_matvec(s.gpu.h, TYPES[c["type"]], s.w.data_ptr(), c["rows"], c["cols"],
                                     s.x.data_ptr(), s.nw.data_ptr() if c["norm"] else None, EPS,
                                     s.y.data_ptr(), 0))
    return s.y


def _exact_matvec(case, seed):
    blocks, x, nw = _matvec_inputs(case, seed)
    x = x.double()[None]
    if case["norm"]:
        x = _rms64(x, nw)
    return _mul64(TYPES[case["type"]], blocks, case["rows"], case["cols"], x)[0]


def _work_matvec(c):
    n = c["rows"] * c["cols"]
    return _mat_bytes(c["type"], n) + 4 * c["rows"] + 8 * c["cols"], 2 * n


# --------------------------------------------------------------------- ffn --
def _ffn_inputs(c, seed):
    H, F, E, qd = c["H"], c["F"], c["E"], c["qd"]
    return dict(wo=_quant(seed, "wo", TYPES[c["attn_type"]], H * qd),
                gate=_quant(seed, "gate", TYPES[c["gate"]], E * F * H),
                up=_quant(seed, "up", TYPES[c["up"]], E * F * H),
                down=_quant(seed, "down", TYPES[c["down"]], E * H * F),
                attn=_normal(seed, "attn", qd, scale=0.7), nw=_norm_w(seed, "norm", H),
                router=_normal(seed, "router", E, H, scale=SIGMA))


def _prepare_ffn(s, c, seed):
    H, F, E, k, qd = c["H"], c["F"], c["E"], c["k"], c["qd"]
    i = _ffn_inputs(c, seed)
    s.attn, s.nw, s.router = i["attn"], i["nw"], i["router"]
    s.wo = _split(s, TYPES[c["attn_type"]], i["wo"], H, qd)
    s.src = {}
    s.mats = []
    for n, rows, cols in (("gate", F, H), ("up", F, H), ("down", H, F)):
        w = _split(s, TYPES[c[n]], i.pop(n), rows, cols, E)
        s.mats.append(w)
        s.src[n] = L.ExpertSrc(w.data_ptr(), _mat_bytes(c[n], F * H), None, 0, None, 0)
    z = lambda *n: torch.empty(*n, device=DEV)  # noqa: E731
    s.x, s.xn, s.logits, s.w, s.gu = z(H), z(H), z(E), z(k), z(2, k, F)
    s.ids = torch.full((64,), -1, dtype=torch.int32, device=DEV)


def _run_ffn(s):
    c, g, lib = s.case, s.gpu.h, s.gpu.lib
    H, F, k = c["H"], c["F"], c["k"]
    L.check(lib.styx_op_matvec(g, TYPES[c["attn_type"]], s.wo.data_ptr(), H, c["qd"],
                               s.attn.data_ptr(), None, 0.0, s.x.data_ptr(), 0))
    L.check(lib.styx_op_router_topk(g, s.x.data_ptr(), s.nw.data_ptr(), EPS, s.router.data_ptr(),
                                    None, c["E"], H, k, 1, None, None, 0, 0, s.xn.data_ptr(),
                                    s.logits.data_ptr(), s.w.data_ptr(), s.ids.data_ptr()))
    L.check(lib.styx_op_moe_gate_up(g, TYPES[c["gate"]], TYPES[c["up"]], C.byref(s.src["gate"]),
                                    C.byref(s.src["up"]), s.ids.data_ptr(), s.xn.data_ptr(),
                                    s.gu.data_ptr(), H, F, k))
    L.check(lib.styx_op_moe_down_reduce(g, TYPES[c["down"]], C.byref(s.src["down"]),
                                        s.ids.data_ptr(), s.w.data_ptr(), s.gu.data_ptr(),
                                        s.x.data_ptr(), H, F, k))
    return {"x": s.x, "xn": s.xn, "logits": s.logits, "weights": s.w}


def _exact_ffn(c, seed):
    i = _ffn_inputs(c, seed)
    H, F = c["H"], c["F"]
    x = _mul64(TYPES[c["attn_type"]], i["wo"], H, c["qd"], i["attn"].double()[None])
    xn = _rms64(x, i["nw"])
    logits = xn @ i["router"].double().T
    y, w, _ = _moe64(xn, logits, c["k"], *((TYPES[c[n]], i[n]) for n in ("gate", "up", "down")), H, F)
    return {"x": (x + y)[0], "xn": xn[0], "logits": logits[0], "weights": w[0]}


def _work_ffn(c):
    H, F, k = c["H"], c["F"], c["k"]
    b = _mat_bytes(c["attn_type"], H * c["qd"]) + 4 * c["E"] * H + 4 * c["qd"] + 16 * H
    b += k * sum(_mat_bytes(c[n], F * H) for n in ("gate", "up", "down"))
    return b, 2 * H * c["qd"] + 2 * c["E"] * H + 6 * k * F * H


# -------------------------------------------------------------------- attn --
PAGE = 512


def _attn_inputs(c, seed):
    n, kvd, qd = c["context"], c["kv"] * c["hd"], c["heads"] * c["hd"]
    pages = -(-n // PAGE)
    order = torch.randperm(pages, generator=_gen(seed, "pages"), device=DEV).to(torch.int32)
    return dict(q=_normal(seed, "q", qd), k=_normal(seed, "k", kvd), v=_normal(seed, "v", kvd),
                qn=_norm_w(seed, "qn", c["hd"]), kn=_norm_w(seed, "kn", c["hd"]),
                kp=_normal(seed, "kp", pages, PAGE, kvd), vp=_normal(seed, "vp", pages, PAGE, kvd),
                pt=order)


def _prepare_attn(s, c, seed):
    s.i = _attn_inputs(c, seed)
    n = c["context"]
    s.rope = _rope_table(c["hd"], n)
    s.pos = torch.tensor([n - 1], dtype=torch.int32, device=DEV)
    s.out = torch.empty(c["heads"] * c["hd"], device=DEV)
    # split as the engine does: chunks of 16 tokens, about 768 workgroups
    s.chunks = min(-(-n // 16), max(16, 768 // c["kv"]))
    s.part = torch.empty(s.gpu.lib.styx_op_attn_part_floats(c["heads"], c["kv"], c["hd"], s.chunks),
                         device=DEV)


def _run_attn(s):
    c, i = s.case, s.i
    norms = (i["qn"].data_ptr(), i["kn"].data_ptr()) if c["norms"] else (None, None)
    L.check(s.gpu.lib.styx_op_attn_decode(
        s.gpu.h, i["q"].data_ptr(), i["k"].data_ptr(), i["v"].data_ptr(), *norms, EPS,
        s.rope.data_ptr(), i["kp"].data_ptr(), i["vp"].data_ptr(), i["pt"].data_ptr(), PAGE,
        s.pos.data_ptr(), s.out.data_ptr(), s.part.data_ptr(), c["heads"], c["kv"], c["hd"], 16,
        s.chunks, 1.0 / math.sqrt(c["hd"])))
    return {"out": s.out, "k": i["kp"], "v": i["vp"]}


def _exact_attn(c, seed):
    i = _attn_inputs(c, seed)
    n, hd, kv, heads = c["context"], c["hd"], c["kv"], c["heads"]
    pos = torch.tensor([n - 1], device=DEV)
    q, k = i["q"].double().view(1, heads, hd), i["k"].double().view(1, kv, hd)
    if c["norms"]:
        q, k = _rms64(q, i["qn"]), _rms64(k, i["kn"])
    q, k = _rope64(q, pos, hd), _rope64(k, pos, hd)
    kp, vp, pt = i["kp"].double(), i["vp"].double(), i["pt"].long()
    kp[pt[(n - 1) // PAGE], (n - 1) % PAGE] = k.view(-1)
    vp[pt[(n - 1) // PAGE], (n - 1) % PAGE] = i["v"].double()
    o = _attend64(q, kp[pt].view(-1, kv, hd)[:n], vp[pt].view(-1, kv, hd)[:n], pos)
    return {"out": o.view(-1), "k": kp, "v": vp}


def _work_attn(c):
    kvd, qd, n = c["kv"] * c["hd"], c["heads"] * c["hd"], c["context"]
    return 8 * n * kvd + 8 * qd + 8 * kvd, 4 * n * qd


# --------------------------------------------------------------- pipelines --
def _dims(n0, n1=1):
    return [n0, n1, 1, 1, 1, n0, n0 * n1, n0 * n1]


def _push_rms(n, rows):
    return struct.pack("<25I", n * rows, *_dims(n, rows), *_dims(n), *_dims(n, rows)) + \
        struct.pack("<I2fi", 0, EPS, 0.0, 0)


def _push_mv(t, rows, cols):
    return struct.pack("<13I", cols, cols // L.BLOCK[t][0], cols, rows, rows * cols, cols, rows,
                       0, 0, 1, 1, 1, 1)


def _push_mv_id(t, rows, cols, k, ne11):
    return struct.pack("<12I", cols, cols // L.BLOCK[t][0], cols, rows, rows * cols, cols,
                       k * rows, 0, k, ne11, 0, 1)


def _push_rope(hd, heads):
    ts = np.float32(ROPE_BASE ** (-2.0 / hd))
    n = [hd, hd * heads, hd * heads]
    return struct.pack("<3I4f2ffI4i3I3I3I3I2I", 2, heads, hd, 1.0, ROPE_BASE, 0.0, 1.0, 0.0, 0.0,
                       ts, 0, 0, 0, 0, 0, 0, 0, 0, hd, heads, 1, *n, *n, 0, 0)


def _push_copy(n):
    return struct.pack("<I8I8II4f8I", n, *_dims(n), *_dims(n), 0, 0, 0, 0, 0, *([0] * 8))


def _layer_inputs(c, seed):
    H, F, E, hd = c["H"], c["F"], c["E"], c["hd"]
    qd, kvd, at = c["heads"] * hd, c["kv"] * hd, TYPES[c["attn_type"]]
    n = c["context"]
    return dict(
        x=_normal(seed, "x", H, scale=0.5), an=_norm_w(seed, "an", H), fn=_norm_w(seed, "fn", H),
        qn=_norm_w(seed, "qn", hd), kn=_norm_w(seed, "kn", hd),
        wq=_quant(seed, "wq", at, qd * H), wk=_quant(seed, "wk", at, kvd * H),
        wv=_quant(seed, "wv", at, kvd * H), wo=_quant(seed, "wo", at, H * qd),
        router=_normal(seed, "router", E, H, scale=SIGMA),
        gate=_quant(seed, "gate", TYPES[c["gate"]], E * F * H),
        up=_quant(seed, "up", TYPES[c["up"]], E * F * H),
        down=_quant(seed, "down", TYPES[c["down"]], E * H * F),
        kc=_normal(seed, "kc", n, kvd), vc=_normal(seed, "vc", n, kvd))


def _prepare_pipelines(s, c, seed):
    H, F, E, k, hd = c["H"], c["F"], c["E"], c["k"], c["hd"]
    heads, kv, n = c["heads"], c["kv"], c["context"]
    qd, kvd, at = heads * hd, kv * hd, TYPES[c["attn_type"]]
    gpu = s.gpu
    b = {}
    for name, v in _layer_inputs(c, seed).items():
        b[name] = gpu.buffer(v.numel() * v.element_size())
        _view(b[name], v.dtype, v.numel()).copy_(v.reshape(-1))
    for name, floats in dict(h=H, q=qd, k=kvd, v=kvd, q1=qd, k1=kvd, q2=qd, k2=kvd, att=qd, o=H,
                             x1=H, logits=E, w=16, g=k * F, u=k * F, d=k * H, none=16).items():
        b[name] = gpu.buffer(floats * 4)
    b["pos"] = gpu.from_numpy(np.array([n - 1] * 4, np.int32))
    b["ids"] = gpu.from_numpy(np.full(64, -1, np.int32))
    b["remap"] = gpu.from_numpy(np.arange(E, dtype=np.uint32))
    b["pmap"] = gpu.from_numpy(np.full(E, L.SKIP, np.uint32))
    s.b = b
    kernels = {}
    s.cmds = []

    def rec(name, binds, push, grid, spec=()):
        key = (name, tuple(spec))
        if key not in kernels:
            kernels[key] = s.own(Kernel(gpu, name, list(spec)))
        arr = (L.Binding * len(binds))()
        for j, x in enumerate(binds):
            buf, off = x if isinstance(x, tuple) else (x, 0)
            arr[j].buf, arr[j].offset, arr[j].range = b[buf].h, off, 2**64 - 1
        gx, gy, gz = (tuple(grid) + (1, 1))[:3]
        s.cmds.append((kernels[key].h, arr, len(binds), C.create_string_buffer(push, len(push)),
                       len(push), gx, gy, gz))

    mv = [(0, 32), (1, 1), (2, 1)]

    def matvec(t, w, x, y, rows, cols):
        rec(f"mul_mat_vec_{_tname(t)}_f32_f32", [w, x, y, "none", "none"], _push_mv(t, rows, cols),
            (rows,), mv)

    def experts(name, w, x, y, rows, cols, ne11):
        t = TYPES[c[name]]
        rec(f"mul_mat_vec_id_{_tname(t)}_f32_f32", [w, x, y, "none", "none", ("ids", 64)],
            _push_mv_id(t, rows, cols, k, ne11), (rows, k), mv)

    rec("rms_norm_f32", ["x", "an", "h"], _push_rms(H, 1), (1,), [(1, 1)])
    matvec(at, "wq", "h", "q", qd, H)
    matvec(at, "wk", "h", "k", kvd, H)
    matvec(at, "wv", "h", "v", kvd, H)
    rec("rms_norm_f32", ["q", "qn", "q1"], _push_rms(hd, heads), (heads,), [(1, 1)])
    rec("rms_norm_f32", ["k", "kn", "k1"], _push_rms(hd, kv), (kv,), [(1, 1)])
    rec("rope_neox_f32", ["q1", "pos", "none", "q2", "none"], _push_rope(hd, heads), (heads, 1))
    rec("rope_neox_f32", ["k1", "pos", "none", "k2", "none"], _push_rope(hd, kv), (kv, 1))
    row = (n - 1) * kvd * 4
    rec("cpy_f32_f32", ["k2", ("kc", row)], _push_copy(kvd), (-(-kvd // 512),))
    rec("cpy_f32_f32", ["v", ("vc", row)], _push_copy(kvd), (-(-kvd // 512),))
    rec("attn_decode_f32", ["q2", "kc", "vc", "att"],
        struct.pack("<4If", n, hd, kvd, heads // kv, 1.0 / math.sqrt(hd)), (heads,))
    matvec(at, "wo", "att", "o", H, qd)
    rec("add_flat_f32", ["x", "o", "x1"], struct.pack("<I", H), (-(-H // 256),))
    rec("rms_norm_f32", ["x1", "fn", "h"], _push_rms(H, 1), (1,), [(1, 1)])
    rec("matvec_strided_f32", ["router", "h", "logits"], struct.pack("<2I", H, H), (E,))
    rec("topk_softmax_f32", ["logits", "w", "ids", "remap", "pmap"], struct.pack("<3I", E, k, 1), (1,))
    experts("gate", "gate", "h", "g", F, H, 1)
    experts("up", "up", "h", "u", F, H, 1)
    rec("swiglu_f32", ["g", "u", "g"], struct.pack("<27I", k * F, *([0] * 26)), (-(-k * F // 512),))
    experts("down", "down", "g", "d", H, F, k)
    rec("moe_reduce_f32", ["d", "w", "x1"], struct.pack("<2I", H, k), (-(-H // 256),))
    s.batch = s.own(Batch(gpu))
    s.out = {"x": _view(b["x1"], torch.float32, H), "k": _view(b["kc"], torch.float32, n, kvd),
             "v": _view(b["vc"], torch.float32, n, kvd)}


def _tname(t):
    return next(n for n, v in TYPES.items() if v == t)


def _run_pipelines(s):
    lib, h = s.gpu.lib, s.batch.h
    L.check(lib.styx_batch_begin(h))
    for k, binds, n, push, ln, gx, gy, gz in s.cmds:
        L.check(lib.styx_batch_dispatch(h, k, binds, n, push, ln, gx, gy, gz, 1))
    L.check(lib.styx_batch_submit(h))
    return s.out


def _exact_pipelines(c, seed):
    i = _layer_inputs(c, seed)
    H, F, hd, heads, kv, n = c["H"], c["F"], c["hd"], c["heads"], c["kv"], c["context"]
    qd, kvd, at = heads * hd, kv * hd, TYPES[c["attn_type"]]
    pos = torch.tensor([n - 1], device=DEV)
    x = i["x"].double()[None]
    h = _rms64(x, i["an"])
    q = _mul64(at, i["wq"], qd, H, h).view(1, heads, hd)
    k = _mul64(at, i["wk"], kvd, H, h).view(1, kv, hd)
    v = _mul64(at, i["wv"], kvd, H, h)
    q, k = _rope64(_rms64(q, i["qn"]), pos, hd), _rope64(_rms64(k, i["kn"]), pos, hd)
    kc, vc = i["kc"].double(), i["vc"].double()
    kc[n - 1], vc[n - 1] = k.view(-1), v[0]
    a = _attend64(q, kc.view(n, kv, hd), vc.view(n, kv, hd), pos).view(1, qd)
    x = x + _mul64(at, i["wo"], H, qd, a)
    h = _rms64(x, i["fn"])
    y, _, _ = _moe64(h, h @ i["router"].double().T, c["k"],
                     *((TYPES[c[m]], i[m]) for m in ("gate", "up", "down")), H, F)
    return {"x": (x + y)[0], "k": kc, "v": vc}


def _work_pipelines(c):
    H, F, k, hd, n = c["H"], c["F"], c["k"], c["hd"], c["context"]
    qd, kvd = c["heads"] * hd, c["kv"] * hd
    b = _mat_bytes(c["attn_type"], 2 * H * (qd + kvd)) + 4 * c["E"] * H + 8 * n * kvd + 20 * H
    b += k * sum(_mat_bytes(c[m], F * H) for m in ("gate", "up", "down"))
    return b, 4 * H * (qd + kvd) + 2 * c["E"] * H + 4 * n * qd + 6 * k * F * H


# ------------------------------------------------------------------- split --
def _prepare_split(s, c, seed):
    s.src = _quant(seed, "w", TYPES[c["type"]], c["experts"] * c["rows"] * c["cols"])
    s.dst = torch.empty(s.src.numel(), dtype=torch.uint8, device=DEV)


def _run_split(s):
    c, t = s.case, TYPES[s.case["type"]]
    L.check(s.gpu.lib.styx_op_to_split(s.gpu.h, t, s.src.data_ptr(), s.dst.data_ptr(),
                                       c["rows"] * c["cols"] // L.BLOCK[t][0], c["experts"]))
    return s.dst


def _exact_split(c, seed):
    return None  # bytes, the same for every implementation of the layout


def _work_split(c):
    return 2 * _mat_bytes(c["type"], c["experts"] * c["rows"] * c["cols"]), 0


# ------------------------------------------------------------------- model --
def _model_types(c, layer):
    mix = [Q4_K, Q5_K, Q6_K]
    return [mix[(layer + r) % 3] if c["mix"] else Q8_0 for r in range(3)]


def _model_specs(c):
    """(name, type, GGUF dims) of every tensor."""
    H, F, E, V = c["H"], c["F"], c["E"], c["vocab"]
    qd, kvd, at = c["heads"] * c["hd"], c["kv"] * c["hd"], TYPES[c["attn_type"]]
    v = [("token_embd.weight", Q8_0, [H, V]), ("output_norm.weight", L.F32, [H]),
         ("output.weight", Q8_0, [H, V])]
    for l in range(c["layers"]):
        g, u, d = _model_types(c, l)
        t = [("attn_norm", L.F32, [H]), ("attn_q_norm", L.F32, [c["hd"]]),
             ("attn_k_norm", L.F32, [c["hd"]]), ("attn_q", at, [H, qd]), ("attn_k", at, [H, kvd]),
             ("attn_v", at, [H, kvd]), ("attn_output", at, [qd, H]), ("ffn_norm", L.F32, [H]),
             ("ffn_gate_inp", L.F32, [H, E]), ("ffn_gate_exps", g, [H, F, E]),
             ("ffn_up_exps", u, [H, F, E]), ("ffn_down_exps", d, [F, H, E])]
        if c["shexp"]:
            t += [("ffn_gate_shexp", g, [H, F]), ("ffn_up_shexp", u, [H, F]),
                  ("ffn_down_shexp", d, [F, H]), ("ffn_gate_inp_shexp", L.F32, [H])]
        v += [(f"blk.{l}.{n}.weight", ty, dims) for n, ty, dims in t]
    return v


def _model_tensor(seed, name, t, dims):
    if t != L.F32:
        return _quant(seed, name, t, math.prod(dims))
    if "norm" in name:
        return _norm_w(seed, name, dims[0])
    return _normal(seed, name, *reversed(dims), scale=SIGMA)


def _prompt(c, seed):
    return torch.randint(0, c["vocab"], (c["prompt"],), generator=_gen(seed, "prompt"), device=DEV)


def _prepare_model(s, c, seed):
    hp = dict(n_layers=c["layers"], n_embd=c["H"], n_heads=c["heads"], n_kv_heads=c["kv"],
              head_dim=c["hd"], n_expert=c["E"], n_expert_used=c["k"], n_ff_exp=c["F"],
              rms_eps=EPS, rope_base=ROPE_BASE)
    root = "/dev/shm" if os.access("/dev/shm", os.W_OK) else None
    with tempfile.TemporaryDirectory(dir=root) as tmp:
        path = os.path.join(tmp, "model.gguf")
        tensors, expert_bytes = [], 0
        for name, t, dims in _model_specs(c):
            a = _model_tensor(seed, name, t, dims).cpu().numpy().reshape(-1)
            expert_bytes += a.nbytes if "exps" in name else 0
            tensors.append((name, t, dims, a.view(np.uint8)))
        gguf_io.write(path, gguf_io.model_metadata(hp), tensors)
        del tensors
        opts = dict(n_ctx=max(512, c["prompt"] + c["new"] + 1))
        if c["host"]:
            # popularity from earlier traffic; the budget holds half the experts
            rng = np.random.default_rng(seed)
            hist = os.path.join(tmp, "hist.csv")
            with open(hist, "w") as f:
                f.write("layer,expert,hits\n")
                for l in range(c["layers"]):
                    for e, h in enumerate(rng.permutation(c["E"])):
                        f.write(f"{l},{e},{1000 // (h + 1)}\n")
            opts.update(expert_budget_mb=(expert_bytes // 2) >> 20, expert_hist=hist)
        s.m = s.own(MoeModel.load(s.gpu, path, **opts), "close")
    s.prompt = _prompt(c, seed).cpu().numpy().astype(np.uint32)


def _run_model(s):
    s.m.reset()
    tokens, _, _ = s.m.generate(s.prompt, s.case["new"])
    logits = s.m.forward_token(int(tokens[-1]))
    return {"tokens": tokens.astype(np.int64), "logits": logits}


def _exact_model(c, seed):
    H, F, hd, heads, kv, V = c["H"], c["F"], c["hd"], c["heads"], c["kv"], c["vocab"]
    qd, kvd, at = heads * hd, kv * hd, TYPES[c["attn_type"]]
    w = {n: (t, _model_tensor(seed, n, t, d)) for n, t, d in _model_specs(c)}
    caches = [(torch.empty(0, kv, hd, dtype=torch.float64, device=DEV),) * 2] * c["layers"]
    per = H // L.BLOCK[Q8_0][0]

    def forward(tokens, first):
        pos = torch.arange(first, first + len(tokens), device=DEV)
        emb = w["token_embd.weight"][1].view(V, per, -1)[tokens]
        x = _dequant64(Q8_0, emb.reshape(len(tokens) * per, -1)).view(len(tokens), H)
        for l in range(c["layers"]):
            t = lambda n: w[f"blk.{l}.{n}.weight"]  # noqa: E731
            h = _rms64(x, t("attn_norm")[1])
            q = _mul64(at, t("attn_q")[1], qd, H, h).view(-1, heads, hd)
            k = _mul64(at, t("attn_k")[1], kvd, H, h).view(-1, kv, hd)
            v = _mul64(at, t("attn_v")[1], kvd, H, h).view(-1, kv, hd)
            q = _rope64(_rms64(q, t("attn_q_norm")[1]), pos, hd)
            k = _rope64(_rms64(k, t("attn_k_norm")[1]), pos, hd)
            kc, vc = torch.cat([caches[l][0], k]), torch.cat([caches[l][1], v])
            caches[l] = (kc, vc)
            a = _attend64(q, kc, vc, pos).view(-1, qd)
            x = x + _mul64(at, t("attn_output")[1], H, qd, a)
            h = _rms64(x, t("ffn_norm")[1])
            y, _, _ = _moe64(h, h @ t("ffn_gate_inp")[1].double().T, c["k"], t("ffn_gate_exps"),
                             t("ffn_up_exps"), t("ffn_down_exps"), H, F)
            x = x + y
            if c["shexp"]:
                y = _swiglu64(h, 0, t("ffn_gate_shexp"), t("ffn_up_shexp"), t("ffn_down_shexp"), H, F)
                sg = torch.sigmoid(h @ t("ffn_gate_inp_shexp")[1].double())
                x = x + y * sg[:, None]
        last = _rms64(x[-1:], w["output_norm.weight"][1])
        return _mul64(Q8_0, w["output.weight"][1], V, H, last)[0]

    logits = forward(_prompt(c, seed), 0)
    tokens = [int(logits.argmax())]
    for i in range(c["new"]):
        logits = forward(torch.tensor(tokens[-1:], device=DEV), c["prompt"] + i)
        tokens.append(int(logits.argmax()))
    return {"tokens": np.array(tokens[:-1], np.int64), "logits": logits}


def _work_model(c):
    H, F, E, k, n = c["H"], c["F"], c["E"], c["k"], c["prompt"]
    qd, kvd = c["heads"] * c["hd"], c["kv"] * c["hd"]
    attn = _mat_bytes(c["attn_type"], 2 * H * (qd + kvd))
    head = _mat_bytes("q8_0", H * c["vocab"])
    met = E * (1.0 - (1.0 - k / E) ** n)  # experts that some prompt token meets
    b = f = 0.0
    for l in range(c["layers"]):
        slab = sum(_n_bytes(t, F * H) for t in _model_types(c, l))
        sh = slab if c["shexp"] else 0
        once = attn + 4 * E * H + sh
        b += once + met * slab + 8 * n * kvd
        b += sum(once + k * slab + 8 * kvd * (n + i + 1) for i in range(c["new"]))
        tok = 4 * H * (qd + kvd) + 2 * E * H + 6 * (k + bool(c["shexp"])) * F * H
        f += tok * (n + c["new"]) + 4 * qd * (n * (n + 1) / 2 + c["new"] * n)
    b += (1 + c["new"]) * (head + 4 * c["vocab"])
    f += (1 + c["new"]) * 2 * H * c["vocab"]
    return b, f


def _n_bytes(t, n):
    el, by = L.BLOCK[t]
    return n // el * by
