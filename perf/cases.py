"""Workloads of the quantized-weight library, as a program that uses it runs them.

Every workload goes through the package's public entry points on data the caller holds on the GPU:
a layer's products one `linear_q` call each, grouped products (`GemvPlan`, `RowsPlan`), the block
codecs, the fake-quantisation pass (`SnapPlan`), GPT-2 generation and Llama / Qwen2 scoring. Sizes
are those of the benchmark's models (GPT-2, Qwen2-0.5B and TinyLlama-1.1B shapes); `draw` gives others of the same ranges.
Weights are packed here, in torch, so that `exact` can compute each result in float64 from the same
blocks without the library.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferrum-gpu_amd"))
import ferrum_hip as fh  # noqa: E402
from ferrum_hip.gguf import F32, STR, U32, Gguf, GgufBuilder, Value  # noqa: E402
from ferrum_hip.gpt2 import GpuGpt2  # noqa: E402
from ferrum_hip.llama import GpuLlama  # noqa: E402

KINDS = {"q8_0": fh.QKind.Q8_0, "q4_0": fh.QKind.Q4_0, "f16": fh.QKind.F16, "fp8_e4m3": fh.QKind.Fp8E4M3,
         "mxfp4": fh.QKind.Fp4, "q2_k": fh.QKind.Q2K}
PATHS = {"auto": fh.QPath.Auto, "tiled": fh.QPath.Tiled, "fast": fh.QPath.TiledFast, "f16": fh.QPath.TiledF16}
# one decoder layer: the model's dim, the stacked q/k/v outputs, the FFN's first product, the FFN's width
GPT2 = {"dim": 768, "qkv": 2304, "up": 3072, "hidden": 3072}
QWEN2 = {"dim": 896, "qkv": 1152, "up": 9728, "hidden": 4864}
LLAMA1B = {"dim": 2048, "qkv": 2560, "up": 11264, "hidden": 5632}


def listed():
    return [
        # one decode step's products of a layer, a call each: latency and launches
        dict(GPT2, name="row1_q8_0_gpt2", family="layer", kind="q8_0", path="auto", rows=1),
        # the same in a format kept as its file rows, wide enough to be bound by memory
        dict(LLAMA1B, name="row1_mxfp4_llama1b", family="layer", kind="mxfp4", path="auto", rows=1),
        # a small batch of sequences decoding together, a call per product
        dict(QWEN2, name="rows24_q8_0_qwen2", family="layer", kind="q8_0", path="auto", rows=24),
        # a prompt through a layer at the reference's product tolerance
        dict(LLAMA1B, name="rows512_q4_0_llama1b", family="layer", kind="q4_0", path="auto", rows=512),
        # a prompt of an odd length on an 8-bit float checkpoint
        dict(LLAMA1B, name="rows300_fp8_llama1b", family="layer", kind="fp8_e4m3", path="auto", rows=300),
        # every layer's one-row products as grouped launches
        dict(QWEN2, name="plan1_q4_0_qwen2", family="plan", kind="q4_0", rows=1, copies=24),
        # the same for eight rows (eight sequences decoding together)
        dict(LLAMA1B, name="plan8_q4_0_llama1b", family="plan", kind="q4_0", rows=8, copies=12),
        # packing a matrix and reading it back
        {"name": "codec_q8_0", "family": "codec", "kind": "q8_0", "rows": 5632, "k": 2048},
        # one fake-quantisation pass of a training step: matrices down their columns, the embedding along
        # its rows, the norm gains copied
        {"name": "snap_llama1b_6_layers", "family": "snap", "layers": 6, "vocab": 32000, "dim": 2048, "kv": 256,
         "hidden": 5632},
        # generation from a short prompt: decode
        {"name": "gpt2_decode", "family": "gpt2", "kind": "q8_0", "dim": 768, "heads": 12, "layers": 12,
         "hidden": 3072, "vocab": 50257, "ctx": 1024, "prompt": 32, "new": 64},
        # a long prompt and its first token: prefill
        {"name": "gpt2_prompt", "family": "gpt2", "kind": "q8_0", "dim": 768, "heads": 12, "layers": 12,
         "hidden": 3072, "vocab": 50257, "ctx": 1024, "prompt": 480, "new": 1},
        # scoring a document
        {"name": "score2048_q4_0_qwen2", "family": "score", "kind": "q4_0", "path": "fast", "dim": 896, "heads": 14,
         "kv_heads": 2, "layers": 24, "hidden": 4864, "vocab": 151936, "tokens": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer_dims(rng, step, odd):
    """A layer between the smallest and the largest of the listed ones; outputs of any count when odd."""
    dim = step * _log_int(rng, 512 // step, 2048 // step)
    hidden = step * max(1, int(dim * rng.uniform(2.0, 5.5)) // step)
    qkv, up = int(dim * rng.uniform(1.2, 3.0)), rng.choice((1, 2)) * hidden
    return {"dim": dim, "qkv": qkv if odd else qkv // 32 * 32, "up": up - (rng.randrange(1, 32) if odd else 0),
            "hidden": hidden}


def draw(rng):
    family = rng.choice(("one row", "few rows", "rows", "other format", "plan", "codec", "snap", "gpt2", "score"))
    kind = rng.choice(("q8_0", "q4_0"))
    odd = rng.random() < 0.5
    if family == "one row":
        return dict(_layer_dims(rng, 32, odd), family="layer", kind=kind, path="auto", rows=1)
    if family == "few rows":
        return dict(_layer_dims(rng, 32, odd), family="layer", kind=kind, path="auto", rows=_log_int(rng, 2, 64))
    if family == "rows":
        return dict(_layer_dims(rng, 32, odd), family="layer", kind=kind, path=rng.choice(("auto", "fast", "f16")),
                    rows=_log_int(rng, 65, 4096))
    if family == "other format":
        kind = rng.choice(("f16", "fp8_e4m3", "mxfp4", "q2_k"))
        return dict(_layer_dims(rng, 256 if kind == "q2_k" else 32, odd), family="layer", kind=kind, path="auto",
                    rows=rng.choice((1, _log_int(rng, 2, 64), _log_int(rng, 65, 1024))))
    if family == "plan":
        return dict(_layer_dims(rng, 32, odd), family="plan", kind=kind, rows=rng.choice((1, _log_int(rng, 2, 64))),
                    copies=_log_int(rng, 2, 16))
    if family == "codec":
        kind = rng.choice(("q8_0", "q4_0", "f16", "fp8_e4m3", "mxfp4", "q2_k"))
        return {"family": "codec", "kind": kind, "rows": _log_int(rng, 33, 5632), "k": 256 * _log_int(rng, 1, 8)}
    if family == "snap":
        return {"family": "snap", "layers": rng.randrange(1, 7), "vocab": _log_int(rng, 500, 32000),
                "dim": 32 * _log_int(rng, 8, 64), "kv": _log_int(rng, 64, 512), "hidden": 32 * _log_int(rng, 16, 176)}
    if family == "gpt2":
        heads = rng.randrange(4, 13)
        short = rng.random() < 0.5
        return {"family": "gpt2", "kind": kind, "dim": 64 * heads, "heads": heads, "layers": rng.randrange(2, 13),
                "hidden": 256 * heads, "vocab": _log_int(rng, 1000, 50257), "ctx": 1024,
                "prompt": _log_int(rng, 1, 48) if short else _log_int(rng, 48, 480),
                "new": _log_int(rng, 16, 64) if short else rng.randrange(1, 9)}
    kv = rng.choice((1, 2, 4))
    heads, hd = kv * rng.randrange(1, 8), 64
    return {"family": "score", "kind": kind, "path": rng.choice(("fast", "tiled")), "dim": heads * hd, "heads": heads,
            "kv_heads": kv, "layers": rng.randrange(2, 13), "hidden": 32 * _log_int(rng, 16, 152),
            "vocab": _log_int(rng, 2000, 151936), "tokens": _log_int(rng, 17, 2048)}


# ---- blocks: f32 rows packed in a block format, and the float64 values of packed rows ----

def _bytes(t):
    return t.contiguous().view(torch.uint8)


def pack(kind, w):
    """Rows [n, k] of f32 in GGUF blocks, [n, k / block elements * block bytes]. Any valid packing serves
    (the values a case computes with are those the blocks hold)."""
    n, k = w.shape
    if kind == "f16":
        return _bytes(w.half()).reshape(n, -1)
    if kind == "q2_k":  # 16 sub-blocks of 4-bit scale and minimum, 2-bit quants, two f16 super-block scales
        b = w.reshape(n, k // 256, 16, 16)
        lo, hi = b.amin(-1).clamp(max=0), b.amax(-1).clamp(min=0)
        d = ((hi - lo).amax(-1) / 45).half()
        m = ((-lo).amax(-1) / 15).half()
        sc = ((hi - lo) / 3 / d.float()[..., None]).round().clamp(1, 15)
        mn = (-lo / m.float()[..., None]).round().clamp(0, 15)
        q = ((b + (m.float()[..., None] * mn)[..., None]) / (d.float()[..., None] * sc)[..., None]).round().clamp(0, 3)
        q = q.to(torch.uint8).reshape(n, k // 256, 2, 4, 32)  # half, plane, element
        qs = (q[:, :, :, 0] | q[:, :, :, 1] << 2 | q[:, :, :, 2] << 4 | q[:, :, :, 3] << 6).reshape(n, -1, 64)
        head = sc.to(torch.uint8) | mn.to(torch.uint8) << 4
        return torch.cat([head, qs, _bytes(d[..., None]), _bytes(m[..., None])], -1).reshape(n, -1)
    b = w.reshape(n, k // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    if kind == "q8_0":
        d = (amax / 127).half()
        q = (b / d.float().clamp(min=1e-12)).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d), _bytes(q)], -1).reshape(n, -1)
    if kind == "q4_0":
        top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
        d = (top / -8).half()
        safe = torch.where(d == 0, torch.ones_like(d), d).float()
        q = (b / safe + 8.5).clamp(0, 15).to(torch.uint8)
        return torch.cat([_bytes(d), q[..., :16] | q[..., 16:] << 4], -1).reshape(n, -1)
    if kind == "fp8_e4m3":
        d = (amax / 448).half()
        q = (b / d.float().clamp(min=1e-12)).clamp(-448, 448).to(torch.float8_e4m3fn)
        return torch.cat([_bytes(d), _bytes(q)], -1).reshape(n, -1)
    e = (torch.floor(torch.log2(amax.clamp(min=1e-30))) + 125).clamp(1, 254)  # mxfp4
    v = (b / torch.exp2(e - 127)).abs()
    steps = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
    q = torch.bucketize(v, steps).to(torch.uint8) | (b < 0).to(torch.uint8) << 3
    return torch.cat([e.to(torch.uint8), q[..., :16] | q[..., 16:] << 4], -1).reshape(n, -1)


def values(kind, rows, k):
    """The float64 values of packed rows, [n, k]."""
    n = rows.shape[0]
    if kind == "f16":
        return rows.view(torch.float16).double()
    if kind == "q2_k":
        b = rows.reshape(n, k // 256, 84)
        d, m = (b[..., i:i + 2].contiguous().view(torch.float16).double() for i in (80, 82))
        qs = b[..., 16:80].reshape(n, -1, 2, 1, 32)
        q = torch.cat([qs >> s & 3 for s in (0, 2, 4, 6)], 3).double().reshape(n, -1, 16, 16)
        return ((d * (b[..., :16] & 15))[..., None] * q - (m * (b[..., :16] >> 4))[..., None]).reshape(n, k)
    b = rows.reshape(n, k // 32, -1)
    if kind == "mxfp4":
        table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                             device=rows.device)
        q = torch.cat([b[..., 1:] & 15, b[..., 1:] >> 4], -1).long()
        return (table[q] * torch.exp2(b[..., :1].double() - 127)).reshape(n, k)
    d, body = b[..., :2].contiguous().view(torch.float16).double(), b[..., 2:].contiguous()
    if kind == "q8_0":
        q = body.view(torch.int8).double()
    elif kind == "q4_0":
        q = torch.cat([body & 15, body >> 4], -1).double() - 8
    else:
        q = body.view(torch.float8_e4m3fn).double()
    return (d * q).reshape(n, k)


def row_bytes(kind, k):
    return {"q8_0": k // 32 * 34, "q4_0": k // 32 * 18, "f16": 2 * k, "fp8_e4m3": k // 32 * 34, "mxfp4": k // 32 * 17,
            "q2_k": k // 256 * 84}[kind]


# ---- shared pieces ----

_gpu = None


def gpu():
    global _gpu
    if _gpu is None:
        _gpu = fh.Gpu(0)
    return _gpu


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) + 1)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


class _Memory:
    """A GpuBuf as torch sees it."""

    def __init__(self, buf, typestr, size):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (size,), "typestr": typestr, "data": (buf.device_ptr(), False),
                                         "version": 3, "strides": None}


def _floats(buf):
    return torch.as_tensor(_Memory(buf, "<f4", buf.len()), device="cuda")


def _uploaded(t):
    """A resident buffer holding the tensor."""
    buf = gpu().zeros(t.numel())
    gpu().sync()
    _floats(buf).copy_(t.reshape(-1))
    torch.cuda.synchronize()
    return buf


def _weight(kind, rows, k, n):
    return fh.upload_qweight(gpu(), KINDS[kind], rows.cpu().numpy(), k, n)


def _shapes(c):
    return [(c["dim"], c["qkv"]), (c["dim"], c["dim"]), (c["dim"], c["up"]), (c["hidden"], c["dim"])]


def _products(c, seed):
    """Packed rows and x of every product of a layer, or of `copies` layers."""
    g = _rng(seed)
    for _ in range(c.get("copies", 1)):
        for k, n in _shapes(c):
            yield k, n, pack(c["kind"], 0.02 * _normal(g, n, k)), _normal(g, c["rows"], k)


def _exact_products(c, seed):
    return [x.double() @ values(c["kind"], rows, k).T for k, n, rows, x in _products(c, seed)]


# ---- GPT-2 and Llama / Qwen2 models ----

def _gpt2_model(c, seed):
    """Tensors of a random-init GPT-2 (normal 0.02, residual projections 0.02 / sqrt(2 layers)): packed rows
    under their GGUF names, vectors, and the prompt."""
    g, d, h, kind = _rng(seed), c["dim"], c["hidden"], c["kind"]
    proj = 0.02 / math.sqrt(2 * c["layers"])
    t = {"token_embd.weight": pack(kind, 0.02 * _normal(g, c["vocab"], d)),
         "position_embd.weight": 0.02 * _normal(g, c["ctx"], d)}
    for i in range(c["layers"]):
        b = f"blk.{i}."
        for name, n, k, s in (("attn_qkv", 3 * d, d, 0.02), ("attn_output", d, d, proj), ("ffn_up", h, d, 0.02),
                              ("ffn_down", d, h, proj)):
            t[b + name + ".weight"] = pack(kind, s * _normal(g, n, k))
            t[b + name + ".bias"] = 0.02 * _normal(g, n)
        for name in ("attn_norm", "ffn_norm"):
            t[b + name + ".weight"] = 1 + 0.1 * _normal(g, d)
            t[b + name + ".bias"] = 0.1 * _normal(g, d)
    t["output_norm.weight"], t["output_norm.bias"] = 1 + 0.1 * _normal(g, d), 0.1 * _normal(g, d)
    prompt = torch.randint(0, c["vocab"], (c["prompt"],), generator=g, device="cuda")
    return t, prompt


def _gguf(meta, tensors, kind, widths):
    b = GgufBuilder()
    for key, tag, v in meta:
        b.meta(key, Value(tag, v))
    for name, t in tensors.items():
        if t.dtype == torch.uint8:
            b.tensor_raw(name, [widths(name), t.shape[0]], int(KINDS[kind]), t.cpu().numpy())
        else:
            b.tensor_f32(name, list(t.shape)[::-1], t.cpu().numpy())
    return Gguf.parse(b.into_bytes())


def _gpt2_exact(c, seed):
    t, prompt = _gpt2_model(c, seed)
    d, heads, L = c["dim"], c["heads"], c["layers"]
    hd = d // heads
    w = {n: values(c["kind"], v, c["hidden"] if "ffn_down" in n else d) if v.dtype == torch.uint8 else v.double()
         for n, v in t.items()}
    keys, vals, done = [None] * L, [None] * L, 0

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, (d,), w[name + ".weight"], w[name + ".bias"], 1e-5)

    def step(ids):
        nonlocal done
        m = ids.numel()
        x = w["token_embd.weight"][ids] + w["position_embd.weight"][done:done + m]
        for i in range(L):
            b = f"blk.{i}."
            lin = lambda a, name: a @ w[b + name + ".weight"].T + w[b + name + ".bias"]  # noqa: E731
            q, k, v = (a.reshape(m, heads, hd).transpose(0, 1) for a in lin(norm(x, b + "attn_norm"), "attn_qkv").split(d, 1))
            keys[i], vals[i] = (a if p is None else torch.cat([p, a], 1) for p, a in ((keys[i], k), (vals[i], v)))
            s = torch.stack([a @ e.T for a, e in zip(q, keys[i])]) / math.sqrt(hd)
            live = torch.arange(done + m, device="cuda")[None] <= torch.arange(done, done + m, device="cuda")[:, None]
            p = s.masked_fill(~live, -math.inf).softmax(-1)
            x = x + lin(torch.stack([a @ e for a, e in zip(p, vals[i])], 1).reshape(m, d), "attn_output")
            u = lin(norm(x, b + "ffn_norm"), "ffn_up")
            x = x + lin(torch.nn.functional.gelu(u, approximate="tanh"), "ffn_down")
        done += m
        return w["token_embd.weight"] @ norm(x[-1], "output_norm")

    logits = step(prompt)
    for _ in range(c["new"]):
        logits = step(logits.argmax().reshape(1))
    return {"tokens": None, "logits": logits.cpu().numpy()}


def _score_model(c, seed):
    """Tensors of a random-init Llama / Qwen2 (uniform, as the package's random models) and the ids."""
    g, d, h, kind = _rng(seed), c["dim"], c["hidden"], c["kind"]
    qd, kvd = c["heads"] * 64, c["kv_heads"] * 64

    def uni(scale, *shape):
        return (2 * torch.rand(*shape, generator=g, device="cuda") - 1) * scale

    qk = 0.5 * math.sqrt(8 / d)
    t = {"token_embd.weight": pack(kind, uni(1.0, c["vocab"], d))}
    for i in range(c["layers"]):
        b = f"blk.{i}."
        for name, n, s in (("attn_q", qd, qk), ("attn_k", kvd, qk), ("attn_v", kvd, 0.5)):
            t[b + name + ".weight"] = pack(kind, uni(s, n, d))
            t[b + name + ".bias"] = uni(0.1, n)
        for name, n, k in (("attn_output", d, qd), ("ffn_gate", h, d), ("ffn_up", h, d), ("ffn_down", d, h)):
            t[b + name + ".weight"] = pack(kind, uni(0.5, n, k))
        for name in ("attn_norm", "ffn_norm"):
            t[b + name + ".weight"] = 1 + uni(0.1, d)
    t["output_norm.weight"] = 1 + uni(0.1, d)
    return t, torch.randint(0, c["vocab"], (c["tokens"],), generator=g, device="cuda")


def _score_exact(c, seed):
    t, ids = _score_model(c, seed)
    d, heads, kvh, n = c["dim"], c["heads"], c["kv_heads"], c["tokens"]
    w = lambda name, k=d: values(c["kind"], t[name], k)  # noqa: E731
    angle = torch.arange(n, device="cuda").double()[:, None] * 1e6 ** (-torch.arange(32, device="cuda").double() / 32)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * t[name].double()

    def rope(a):
        a = a.reshape(n, -1, 64)
        lo, hi = a[..., :32], a[..., 32:]
        return torch.cat([lo * cos - hi * sin, lo * sin + hi * cos], -1)

    x = values(c["kind"], t["token_embd.weight"][ids], d)
    dead = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for i in range(c["layers"]):
        b = f"blk.{i}."
        h = norm(x, b + "attn_norm.weight")
        q, k, v = (h @ w(b + m + ".weight").T + t[b + m + ".bias"].double() for m in ("attn_q", "attn_k", "attn_v"))
        q, k, v = rope(q), rope(k), v.reshape(n, kvh, 64)
        o = []
        for a in range(heads):
            s = (q[:, a] @ k[:, a * kvh // heads].T / 8).masked_fill_(dead, -math.inf)
            o.append(s.softmax(-1) @ v[:, a * kvh // heads])
        x = x + torch.cat(o, 1) @ w(b + "attn_output.weight", heads * 64).T
        h = norm(x, b + "ffn_norm.weight")
        act = torch.nn.functional.silu(h @ w(b + "ffn_gate.weight").T) * (h @ w(b + "ffn_up.weight").T)
        x = x + act @ w(b + "ffn_down.weight", c["hidden"]).T
    h, out, first = norm(x, "output_norm.weight")[:-1], [], []
    head = w("token_embd.weight")
    for r in range(0, n - 1, 256):
        logits, want = h[r:r + 256] @ head.T, ids[r + 1:r + 257]
        want = want[:logits.shape[0]]
        out.append(logits.log_softmax(-1).gather(1, want[:, None])[:, 0])
        first.append((logits.argmax(-1) == want).double())
    return [torch.cat(out), torch.cat(first)]


# ---- fake quantisation ----

def _snap_tensors(c, seed):
    """(mode, shape, values) of every parameter of a Llama-style model."""
    g, d = _rng(seed), c["dim"]
    for _ in range(c["layers"]):
        for k, n in ((d, d), (d, c["kv"]), (d, c["kv"]), (d, d), (d, c["hidden"]), (d, c["hidden"]), (c["hidden"], d)):
            yield fh.SNAP_COLS, (k, n), 0.02 * _normal(g, k * n)
        yield fh.SNAP_COPY, d, 1 + 0.1 * _normal(g, d)
    yield fh.SNAP_ROWS, d, 0.02 * _normal(g, c["vocab"] * d)


# ---- the interface ----

def prepare(case, seed):
    c, family = dict(case), case["family"]
    if family == "layer":
        items = []
        for k, n, rows, x in _products(c, seed):
            items.append((_weight(c["kind"], rows, k, n), x, torch.empty(c["rows"], n, device="cuda")))
        torch.cuda.synchronize()
        return {"family": family, "path": PATHS[c["path"]], "rows": c["rows"], "items": items,
                "out": [y for _, _, y in items]}
    if family == "plan":
        ys = [torch.empty(c["copies"], c["rows"], n, device="cuda") for _, n in _shapes(c)]
        xs, problems = [], []
        for i, (k, n, rows, x) in enumerate(_products(c, seed)):
            xs.append(x)
            p = (_weight(c["kind"], rows, k, n), x.data_ptr(), ys[i % 4][i // 4].data_ptr())
            problems.append(p if c["rows"] == 1 else p + (c["rows"],))
        torch.cuda.synchronize()
        plan = (fh.GemvPlan if c["rows"] == 1 else fh.RowsPlan)(gpu(), problems)
        return {"family": family, "plan": plan, "x": xs, "out": ys}
    if family == "codec":
        kind, n = KINDS[c["kind"]], c["rows"] * c["k"]
        src = _uploaded(0.02 * _normal(_rng(seed), n))
        packed, dst = gpu().bytes_zeros(fh.nbytes(kind, n)), gpu().zeros(n)
        gpu().sync()
        view = torch.as_tensor(_Memory(packed, "|u1", packed.nbytes()), device="cuda")
        return {"family": family, "kind": kind, "n": n, "src": src, "packed": packed, "dst": dst,
                "out": [view, _floats(dst)]}
    if family == "snap":
        problems, out = [], []
        for mode, shape, v in _snap_tensors(c, seed):
            dst = gpu().zeros(v.numel())
            problems.append((mode, _uploaded(v), dst, shape))
            out.append(_floats(dst))
        gpu().sync()
        return {"family": family, "plan": fh.SnapPlan(gpu(), problems), "out": out}
    if family == "gpt2":
        t, prompt = _gpt2_model(c, seed)
        meta = [("general.architecture", STR, "gpt2")]
        meta += [("gpt2." + key, U32, c[field]) for key, field in (
            ("context_length", "ctx"), ("embedding_length", "dim"), ("block_count", "layers"),
            ("feed_forward_length", "hidden"), ("attention.head_count", "heads"))]
        meta.append(("gpt2.attention.layer_norm_epsilon", F32, float(np.float32(1e-5))))
        g = _gguf(meta, t, c["kind"], lambda n: c["hidden"] if "ffn_down" in n else c["dim"])
        return {"family": family, "model": GpuGpt2.from_gguf(gpu(), g), "prompt": prompt.cpu().numpy().astype(np.int32),
                "new": c["new"]}
    t, ids = _score_model(c, seed)
    meta = [("general.architecture", STR, "qwen2")]
    meta += [("qwen2." + key, U32, v) for key, v in (
        ("context_length", max(2048, c["tokens"])), ("embedding_length", c["dim"]), ("block_count", c["layers"]),
        ("feed_forward_length", c["hidden"]), ("attention.head_count", c["heads"]),
        ("attention.head_count_kv", c["kv_heads"]), ("attention.key_length", 64), ("rope.dimension_count", 64))]
    meta += [("qwen2.rope.freq_base", F32, 1e6), ("qwen2.attention.layer_norm_rms_epsilon", F32, float(np.float32(1e-6)))]
    g = _gguf(meta, t, c["kind"], lambda n: c["hidden"] if "ffn_down" in n else
              c["heads"] * 64 if "attn_output" in n else c["dim"])
    model = GpuLlama.from_gguf(gpu(), g, PATHS[c["path"]])
    buf, out = _uploaded(ids.to(torch.int32).view(torch.float32)), gpu().zeros(2 * (c["tokens"] - 1))
    gpu().sync()
    return {"family": family, "model": model, "ids": buf, "n": c["tokens"], "dst": out,
            "out": list(_floats(out).view(-1, 2).unbind(1))}


def run(state):
    family = state["family"]
    if family == "layer":
        for w, x, y in state["items"]:
            fh.linear_q_ptr(gpu(), x.data_ptr(), w, y.data_ptr(), state["rows"], state["path"])
    elif family == "codec":
        fh.encode(gpu(), state["kind"], state["src"], state["n"], state["packed"])
        fh.decode(gpu(), state["kind"], state["packed"], state["n"], state["dst"])
    elif family == "gpt2":
        model = state["model"]
        model.reset()
        tokens = model.generate(state["prompt"], state["new"])
        return {"tokens": np.array(tokens), "logits": model.feed(tokens[-1])}
    elif family == "score":
        state["model"].score_device(state["ids"], state["n"], state["dst"])
    else:
        state["plan"].run()
    return state["out"]


def work(case):
    c, family = case, case["family"]
    if family in ("layer", "plan"):
        copies, m = c.get("copies", 1), c["rows"]
        return {"bytes": copies * sum(n * row_bytes(c["kind"], k) + 4 * m * (k + n) for k, n in _shapes(c)),
                "flops": copies * sum(2 * m * k * n for k, n in _shapes(c))}
    if family == "codec":  # encode: f32 in, blocks out; decode: the reverse
        n = c["rows"] * c["k"]
        return {"bytes": 2 * (4 * n + c["rows"] * row_bytes(c["kind"], c["k"])), "flops": 0}
    d, h = c["dim"], c["hidden"]
    if family == "snap":
        layer = 2 * d * d + 2 * d * c["kv"] + 3 * d * h + d
        return {"bytes": 8 * (c["layers"] * layer + c["vocab"] * d), "flops": 0}
    if family == "gpt2":
        layer = row_bytes(c["kind"], d) * (4 * d + h) + d * row_bytes(c["kind"], h)
        head, steps, kv = c["vocab"] * row_bytes(c["kind"], d), c["new"] + 1, 8 * d * c["layers"]
        # the prompt reads the weights once, each further token once, and every token's k and v once per later token
        seen = sum(range(c["prompt"], c["prompt"] + c["new"]))
        total = c["prompt"] + c["new"]
        return {"bytes": steps * (c["layers"] * layer + head) + kv * (total + seen),
                "flops": 2 * total * c["layers"] * (4 * d * d + 2 * d * h) + 2 * steps * c["vocab"] * d
                + 2 * c["layers"] * d * total * total}
    qd, kvd, n = c["heads"] * 64, c["kv_heads"] * 64, c["tokens"]
    layer = d * (qd + 2 * kvd) + qd * d + 3 * d * h
    return {"bytes": (c["layers"] * layer + c["vocab"] * d) * row_bytes(c["kind"], 32) / 32 + 12 * n,
            "flops": 2 * n * (c["layers"] * layer + c["vocab"] * d) + 2 * c["layers"] * qd * n * (n + 1)}


def tolerance(case):
    family = case["family"]
    if family in ("codec", "snap"):
        return "exact"
    # about four times the error against float64 that the measured paths show
    if family == "gpt2":  # 2.4e-7
        return {"rel": 1.5e-6, "max": 2e-5}
    if family == "score":  # log-probabilities after every layer's products: 2.4e-5 and 1.2e-6
        return {"rel": 1e-4, "max": 2e-3} if case["path"] == "fast" else {"rel": 1e-5, "max": 2e-4}
    if family == "layer" and case["path"] == "f16":  # both operands round to 11 bits
        return {"rel": 1.5e-3, "max": 1e-2}
    if family == "layer" and case["path"] == "fast":  # 7.4e-6
        return {"rel": 3e-5, "max": 3e-4}
    return {"rel": 1e-6, "max": 1e-5}  # 0.7e-7 to 1.8e-7


def exact(case, seed):
    c, family = case, case["family"]
    if family == "layer":
        return [y for y in _exact_products(c, seed)]
    if family == "plan":
        out = [torch.empty(c["copies"], c["rows"], n, device="cuda", dtype=torch.float64) for _, n in _shapes(c)]
        for i, (k, n, rows, x) in enumerate(_products(c, seed)):
            out[i % 4][i // 4] = x.double() @ values(c["kind"], rows, k).T
        return out
    if family == "gpt2":
        return _gpt2_exact(c, seed)
    if family == "score":
        return _score_exact(c, seed)
    return None  # bytes, and values on the blocks' grid: whole numbers
