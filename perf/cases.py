"""The matrix-multiplication work a user of this framework has it do, as cases
that can be timed and checked: decode steps, the lm_head, prefill blocks from
a short prompt's to a full block's, and the MoE layer from a decode batch's
tokens to a full block's.

A case names a path and its rows.  Every path goes through the package's
public interface (Gpu, Engine, MoeLayer): kernels chosen by the engine for
the shape, once per process as at a model's load, then launched on the
library's buffers.  Prefill rows run on the kernels of their bucket (the
smallest of Engine.buckets that holds them), decode rows on those of 1, 4 or
8 rows, MoE tokens on a layer of 64 or 2048 rows.

The shapes: a 4B-class dense layer (hidden 2560, 16 q heads and 4 kv heads of
256, MLP 9216, vocabulary 151936), the 27B-class down projection (17408 to
5120) and fused QKV (5120 to 7168), a single 1024 to 3584 GEMM, and a
35B-A3B-class sparse layer (hidden 2048, 256 experts, top 8, intermediate
512).  Activations ~ N(0, 1), weights ~ N(0, 0.02), scores ~ N(0, 1), bf16.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "herbert-metal-bf16_amd"))
import herbert_hip as hb  # noqa: E402

H, Q, QKV, INTER, VOCAB = 2560, 4096, 4608, 9216, 151936
QKV_WIDE = 10240  # the gated fused QKV: q, its gate, k, v
EXPERTS, TOP_K, MH, MI = 256, 8, 2048, 512
EPS = 1e-6


def listed():
    return [
        # One sequence decoding: a layer's projections with the norms, the
        # SwiGLU and the residual adds in them; launches and latency count.
        {"name": "decode_layer_m1", "path": "decode_fused", "m": 1},
        # A batch of eight sequences decoding, norms and SwiGLU apart.
        {"name": "decode_layer_m8", "path": "decode", "m": 8},
        # Four sequences' logits: the largest matrix of a decode step.
        {"name": "lm_head_m4", "path": "head", "m": 4},
        # A chat turn of a few words: the MLP half of a layer, 57 rows.
        {"name": "mlp_m57", "path": "mlp", "m": 57},
        # A paragraph: the attention half's projections, 200 rows.
        {"name": "attn_m200", "path": "attn", "m": 200},
        # One GEMM of 512 x 1024 x 3584, the benchmark's first shape.
        {"name": "gemm_m512", "path": "gemm", "k": 1024, "n": 3584, "out": "Bf16", "m": 512},
        # A page: the MLP half over a block of 512 rows.
        {"name": "mlp_m512", "path": "mlp", "m": 512},
        # A long prompt's full block through a layer's four GEMMs.
        {"name": "layer_m2048", "path": "layer", "m": 2048},
        # The last, ragged block of a long prompt on the 27B-class down.
        {"name": "down27_m1100", "path": "gemm", "k": 17408, "n": 5120, "out": "Residual", "m": 1100},
        # The sparse layer: a decode batch, a short prompt, a full block.
        {"name": "moe_t8", "path": "moe", "t": 8},
        {"name": "moe_t50", "path": "moe", "t": 50},
        {"name": "moe_t2048", "path": "moe", "t": 2048},
    ]


def draw(rng):
    path = rng.choice(["decode_fused", "decode", "head", "mlp", "attn", "layer", "gemm", "gemm", "moe", "moe"])
    if path == "moe":
        return {"path": path, "t": int(round(math.exp(rng.uniform(math.log(1), math.log(2047)))))}
    if path == "decode_fused":  # with one sequence or up to four
        return {"path": path, "m": rng.randint(2, 4)}
    if path in ("decode", "head"):
        return {"path": path, "m": rng.choice([1, 2, 3, 5, 6, 7])}
    m = int(round(math.exp(rng.uniform(math.log(9), math.log(2047)))))
    if path == "gemm":
        k, n, out = rng.choice([(1024, 3584, "Bf16"), (1024, 3584, "F32"), (2560, 4608, "Bf16"), (2560, 10240, "Bf16"),
                                (5120, 7168, "Bf16"), (17408, 5120, "Residual")])
        return {"path": path, "k": k, "n": n, "out": out, "m": m}
    return {"path": path, "m": m}


# ---- the library and its buffers ----

_lib = {}


def _open():
    """The process's device context and its engine."""
    if not _lib:
        gpu = hb.Gpu.open()
        _lib["gpu"], _lib["engine"] = gpu, hb.Engine(gpu)
    return _lib["gpu"], _lib["engine"]


_TYPES = {torch.bfloat16: ("<i2", torch.int16), torch.float32: ("<f4", torch.float32), torch.int32: ("<i4", torch.int32)}


class _View:
    """A library buffer as an array torch can wrap; holds on to its owner."""

    def __init__(self, owner, buf, shape, dtype):
        p = ctypes.c_void_p()
        hb.check(hb.lib.hb_buffer_ptr(owner.gpu.h, buf, ctypes.byref(p)))
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": _TYPES[dtype][0], "data": (p.value, False),
                                         "version": 2}


def _tensor(owner, buf, shape, dtype=torch.bfloat16):
    t = torch.as_tensor(_View(owner, buf, shape, dtype), device="cuda")
    return t.view(dtype)


class _Buf:
    """A device buffer of the library and the torch tensor over it."""

    def __init__(self, gpu, shape, dtype=torch.bfloat16):
        self.gpu = gpu
        self.id = gpu.alloc(int(np.prod(shape)) * torch.empty(0, dtype=dtype).element_size())
        self.shape, self.dtype = shape, dtype

    @property
    def t(self):
        return _tensor(self, self.id, self.shape, self.dtype)

    def __del__(self):
        self.gpu.free(self.id)


class _Moe:
    """A MoeLayer that gives its buffers back."""

    def __init__(self, gpu, layer, weights):
        self.gpu, self.layer, self.weights = gpu, layer, weights

    def __del__(self):
        self.layer.free()


# ---- the inputs, from the seed ----

def _weights_of(case):
    """{name: shape} of the case's weights."""
    p = case["path"]
    if p == "gemm":
        return {"w": (case["n"], case["k"])}
    if p == "head":
        return {"w": (VOCAB, H)}
    if p == "moe":
        return {"gate_up": (EXPERTS, 2 * MI, MH), "down": (EXPERTS, MH, MI)}
    attn = {"input_norm": (H,), "qkv": (QKV_WIDE if p == "attn" else QKV, H), "o": (H, Q)}
    mlp = {"post_norm": (H,), "gate_up": (2 * INTER, H), "down": (H, INTER)}
    return attn if p == "attn" else mlp if p == "mlp" else {**attn, **mlp}


def _inputs_of(case):
    """{name: shape} of what the call brings besides the weights."""
    p = case["path"]
    if p == "moe":
        return {"x": (case["t"], MH), "scores": (case["t"], EXPERTS)}
    m = case["m"]
    if p == "gemm":
        d = {"x": (m, case["k"])}
        if case["out"] == "Residual":
            d["y"] = (m, case["n"])
        return d
    if p in ("head", "mlp"):
        return {"x": (m, H)}
    return {"x": (m, H), "ao": (m, Q)}


def _draws(case, seed):
    """(name, values) of every weight and input in turn, bf16 on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2654435761 % (1 << 62))
    for name, shape in _weights_of(case).items():
        # The norms' weights are stored less one (plus_one).
        yield name, torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0, 0.1 if "norm" in name else 0.02, generator=g)
    for name, shape in _inputs_of(case).items():
        yield name, torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0, 1, generator=g)


def _bucket(engine, m):
    return min(b for b in engine.buckets() if b >= m)


def _mv_rows(m):
    return 1 if m == 1 else 4 if m <= 4 else 8


# ---- the case in the library's hands ----

def prepare(case, seed):
    gpu, eng = _open()
    if case["path"] == "moe":
        return _prepare_moe(gpu, eng, case, seed)
    p, m = case["path"], case["m"]
    decode = p in ("decode", "decode_fused", "head")
    # Row buffers hold the rows the kernels were chosen for.
    rows = _mv_rows(m) if decode else _bucket(eng, m)
    bufs = {}

    def buf(name, shape, dtype=torch.bfloat16):
        bufs[name] = _Buf(gpu, shape, dtype)
        return bufs[name]

    for name, v in _draws(case, seed):
        if name in _inputs_of(case):
            buf(name, (rows, v.shape[1])).t.zero_()[:m].copy_(v)
        else:
            buf(name, tuple(v.shape)).t.copy_(v)
    buf("state", (4,), torch.int32).t.copy_(torch.tensor([0, 0, 0, rows], dtype=torch.int32))
    if p not in ("gemm", "head"):
        buf("xn", (rows, H))
    if p in ("decode", "decode_fused", "attn", "layer"):
        buf("qkv_out", (rows, _weights_of(case)["qkv"][0]))
    if p in ("decode", "decode_fused", "mlp", "layer"):
        buf("gu", (rows, 2 * INTER))
        buf("h", (rows, INTER))
    if p == "gemm" and "y" not in bufs:
        buf("y", (rows, case["n"]), torch.float32 if case["out"] == "F32" else torch.bfloat16)
    if p == "head":
        buf("logits", (rows, VOCAB))
    torch.cuda.synchronize()
    b = {k: hb.r(v.id) for k, v in bufs.items()}
    keep = bufs["x"].t.clone(), bufs["y"].t.clone() if "y" in bufs else None
    torch.cuda.synchronize()
    norm = gpu.pipeline(hb.rmsnorm(H, EPS, True)) if p not in ("gemm", "head", "decode_fused") else -1
    steps = []
    out = {}

    def gemm(k, n, o, w, x, y):
        kern = eng.gemm(k, n, o, b["state"], b[w], b[x], b[y], rows)
        steps.append((kern, [b["state"], b[w], b[x], b[y], b["state"], b["state"]], m))

    def mv(k, n, o, w, x, y):
        kern = eng.mv(k, n, o, rows, [b[w]], b[x], b[y])
        steps.append((kern, [b[w], b[x], b[y]], m))

    def mv_norm(k, n, o, w, x, y, nw):
        kern = eng.mv_fused(k, n, o, rows, [b[w]], b[x], b[y], xsrc=hb.XSrc.Norm, eps=EPS, plus_one=True, norm_w=b[nw])
        steps.append((kern, [b[w], b[x], b[y], b[nw]], m))

    def normed(w):
        steps.append((norm, [b["x"], b[w], b["xn"]], m))

    if p == "gemm":
        gemm(case["k"], case["n"], hb.Out[case["out"]], "w", "x", "y")
        out["y"] = bufs["y"].t[:m]
    elif p == "head":
        mv(H, VOCAB, hb.Out.Bf16, "w", "x", "logits")
        out["logits"] = bufs["logits"].t[:m]
    if "input_norm" in b:
        n = _weights_of(case)["qkv"][0]
        if p == "decode_fused":
            mv_norm(H, n, hb.Out.Bf16, "qkv", "x", "qkv_out", "input_norm")
            mv(Q, H, hb.Out.Residual, "o", "ao", "x")
        elif p == "decode":
            normed("input_norm")
            mv(H, n, hb.Out.Bf16, "qkv", "xn", "qkv_out")
            mv(Q, H, hb.Out.Residual, "o", "ao", "x")
        else:
            normed("input_norm")
            gemm(H, n, hb.Out.Bf16, "qkv", "xn", "qkv_out")
            gemm(Q, H, hb.Out.Residual, "o", "ao", "x")
        out["qkv"], out["x"] = bufs["qkv_out"].t[:m], bufs["x"].t[:m]
    if "post_norm" in b:
        if p == "decode_fused":
            mv_norm(H, 2 * INTER, hb.Out.Swiglu, "gate_up", "x", "h", "post_norm")
            mv(INTER, H, hb.Out.Residual, "down", "h", "x")
        elif p == "decode":
            normed("post_norm")
            mv(H, 2 * INTER, hb.Out.Bf16, "gate_up", "xn", "gu")
            steps.append((gpu.pipeline(hb.swiglu_rows(INTER)), [b["gu"], b["h"]], m))
            mv(INTER, H, hb.Out.Residual, "down", "h", "x")
        else:
            normed("post_norm")
            gk, sk = eng.gate_up(H, INTER, b["state"], b["gate_up"], b["xn"], b["gu"], b["h"], rows)
            st = b["state"]
            steps.append((gk, [st, b["gate_up"], b["xn"], b["gu" if sk >= 0 else "h"], st, st], m))
            if sk >= 0:
                steps.append((sk, [b["gu"], b["h"]], m))
            gemm(INTER, H, hb.Out.Residual, "down", "h", "x")
        out["h"], out["x"] = bufs["h"].t[:m], bufs["x"].t[:m]
    gpu.sync()
    # The selection's timed runs added into the residual rows: as they were.
    bufs["x"].t.copy_(keep[0])
    if keep[1] is not None:
        bufs["y"].t.copy_(keep[1])
    bufs["state"].t.copy_(torch.tensor([0, 0, 0, m], dtype=torch.int32))
    torch.cuda.synchronize()
    return {"gpu": gpu, "steps": steps, "out": out, "bufs": bufs}


def _prepare_moe(gpu, eng, case, seed):
    t = case["t"]
    rows = 64 if t <= 64 else 2048
    v, weights = {}, {}
    for name, x in _draws(case, seed):
        if name in _inputs_of(case):
            v[name] = x
        else:
            weights[name] = _Buf(gpu, tuple(x.shape))
            weights[name].t.copy_(x)
    # The engine times the experts on a route of the layer's whole block:
    # the call's tokens, repeated to fill it.
    fill = {k: x.repeat(-(-rows // t), 1)[:rows] for k, x in v.items()}
    if t < rows:  # other tokens' scores after the call's own
        g = torch.Generator(device="cuda")
        g.manual_seed(seed + 1)
        fill["scores"][t:].normal_(0, 1, generator=g)
    torch.cuda.synchronize()
    host = {k: x.view(torch.int16).cpu().numpy().view(np.uint16) for k, x in fill.items()}
    layer = _Moe(gpu, hb.MoeLayer(gpu, eng, EXPERTS, TOP_K, MH, MI, rows, weights["gate_up"].id, weights["down"].id,
                                  scores=host["scores"], x=host["x"]), weights)
    gpu.upload(layer.layer.buf["state"], np.array([0, 0, 0, t], np.uint32))
    gpu.sync()
    return {"moe": layer, "m": t, "out": {"out": _tensor(layer, layer.layer.buf["out"], (t, MH))}}


def run(state):
    if "moe" in state:
        state["moe"].layer.run(state["m"])
        return state["out"]
    gpu = state["gpu"]
    for kern, ranges, m in state["steps"]:
        gpu.launch(kern, ranges, m)
    return state["out"]


# ---- what a pass cannot do without ----

def work(case):
    p = case["path"]
    if p == "moe":
        t = case["t"]
        hit = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** t)  # experts with rows
        per = 3 * MI * MH
        return {"bytes": 2.0 * (hit * per + 2 * t * MH + t * EXPERTS), "flops": 2.0 * t * TOP_K * per}
    m = case["m"]
    weights = _weights_of(case)
    flops = sum(2.0 * m * s[0] * s[1] for s in weights.values() if len(s) == 2)
    bytes_ = 2.0 * sum(np.prod(s) for s in weights.values()) + 2.0 * sum(np.prod(s) for s in _inputs_of(case).values())
    # The outputs: written once (the residual's old values are an input).
    if p == "gemm":
        bytes_ += m * case["n"] * (4.0 if case["out"] == "F32" else 2.0)
    elif p == "head":
        bytes_ += 2.0 * m * VOCAB
    else:
        if "qkv" in weights:
            bytes_ += 2.0 * m * weights["qkv"][0]
        if "down" in weights:
            bytes_ += 2.0 * m * INTER
        bytes_ += 2.0 * m * H
    return {"bytes": float(bytes_), "flops": flops}


def tolerance(case):
    p = case["path"]
    # Each about four times what the same path differs by when its sums run
    # in another order (the sequential VALU GEMM and K split four ways in
    # the matvec, against the chosen kernels).
    if p == "gemm" and case["out"] == "F32":
        return {"rel": 1.2e-6, "max": 1e-5}  # seen 2.8e-7, 2.3e-6
    # One bf16 rounding: a few outputs in ten thousand land on its other side.
    if p in ("gemm", "head"):
        return {"rel": 4e-4, "max": 6e-2}  # seen 9e-5, 1.5e-2
    # The chained paths carry such roundings through a norm, a SwiGLU and a
    # second matrix, the sparse layer through its eight rounded adds.
    return {"rel": 3e-3, "max": 8e-2}  # seen 7e-4, 2e-2


# ---- the same in 64 bits, by torch ----

def _mm(x, w):
    return x @ w.double().T


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (w.double() + 1.0)


def _swiglu(gu):
    g, u = gu.chunk(2, -1)
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    v = dict(_draws(case, seed))
    x = v["x"].double()
    p = case["path"]
    if p == "moe":
        probs = torch.softmax(v["scores"].double(), -1)
        # The k best, the lower expert where two are equal.
        top = torch.sort(probs, dim=-1, descending=True, stable=True)
        ids, w = top.indices[:, :TOP_K], top.values[:, :TOP_K]
        w = w / w.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        for e in ids.unique().tolist():
            tok, slot = (ids == e).nonzero(as_tuple=True)
            y = _mm(_swiglu(_mm(x[tok], v["gate_up"][e])), v["down"][e])
            out.index_add_(0, tok, y * w[tok, slot][:, None])
        return {"out": out}
    if p == "gemm":
        y = _mm(x, v["w"])
        return {"y": y + v["y"].double() if case["out"] == "Residual" else y}
    if p == "head":
        return {"logits": _mm(x, v["w"])}
    out = {}
    if "qkv" in v:
        out["qkv"] = _mm(_rms(x, v["input_norm"]), v["qkv"])
        x = x + _mm(v["ao"].double(), v["o"])
    if "down" in v:
        out["h"] = _swiglu(_mm(_rms(x, v["post_norm"]), v["gate_up"]))
        x = x + _mm(out["h"], v["down"])
    out["x"] = x
    return out
