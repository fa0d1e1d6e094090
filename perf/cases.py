"""The work this framework is used for, as cases that can be timed.

Every case goes through the public entry points the way a model's program
calls them, on the GPU, with the buffers such a program keeps (weights, the
KV cache, outputs, RoPE tables, a captured graph).  Kinds:

* ``gqa``     -- ``attention_gqa`` on one prompt, the drop-in call of the
                 reference's models;
* ``prefill`` -- ``flash_attention`` over a batch of prompts;
* ``prompt``  -- one layer's attention sub-block for a prompt through
                 ``GpuKVCache.attention``: RoPE, cache write, attention in the
                 model's (seq, heads * d_k) rows;
* ``decode``  -- ``decode_step`` for a batch of sequences of unequal length:
                 RoPE, cache append, attention over the cache;
* ``mlp``     -- residual add + RMSNorm, gate / up, SwiGLU, down, residual add;
* ``layer``   -- a whole decoder layer for a prompt;
* ``token``   -- one decoded token of a model at batch 1, embedding row to
                 logits, as a captured graph that a generate loop replays;
* ``sample``  -- the next token of every sequence from its logits.

Inputs are made on the GPU from the seed.  Sequence lengths of a decode batch
come from the case itself, so that its work does not depend on the seed.
"""

from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "triton-llm_amd"))

from triton_llm import gpu  # noqa: E402
from triton_llm.kernels import (  # noqa: E402
    add, add_rms_norm, attention_gqa, decode_step, decode_workspace, flash_attention, gemm, gemm_grouped,
    precompute_cos_sin, rms_norm, sample_rows, swiglu)
from triton_llm.kv_cache import GpuKVCache  # noqa: E402

TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
STORE = {"float32": np.dtype(np.float32), "float16": np.dtype(np.float16), "bfloat16": gpu.bfloat16}
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}

# Heads of the models the framework names, and their widths.
HEADS = {"gpt2": (12, 12, 64), "smollm2-135m": (9, 3, 64), "smollm2-360m": (15, 5, 64), "llama3.2-3b": (24, 8, 128)}
WIDTH = {"smollm2-360m": (960, 2560), "llama3.2-3b": (3072, 8192)}  # (n_embd, intermediate)
THETA = {"smollm2-135m": 1e4, "smollm2-360m": 1e4, "llama3.2-3b": 5e5}


def listed():
    return [
        # GPT-2's 128-token prompt in the reference's own type: the smallest call a model makes.
        {"name": "gpt2-prompt-fp32", "kind": "gqa", "model": "gpt2", "dtype": "float32", "seq": 128},
        # A small serving batch on GPT-2: short caches, latency counts.
        {"name": "gpt2-decode-fp16", "kind": "decode", "model": "gpt2", "dtype": "float16", "batch": 8,
         "max_ctx": 1024, "lo": 1, "hi": 1023, "lens": 1},
        # SmolLM2-135M's prompts, four sequences at once.
        {"name": "smollm2-135m-prefill-bf16", "kind": "prefill", "model": "smollm2-135m", "dtype": "bfloat16",
         "batch": 4, "seq": 2048, "causal": True},
        # An ordinary serving batch: 32 sequences with up to 8192 cached tokens.
        {"name": "smollm2-360m-decode-bf16", "kind": "decode", "model": "smollm2-360m", "dtype": "bfloat16",
         "batch": 32, "max_ctx": 8192, "lo": 512, "hi": 8191, "lens": 3},
        # A long prompt, Llama-3.2-3B heads.
        {"name": "llama-prefill-8192-bf16", "kind": "prefill", "model": "llama3.2-3b", "dtype": "bfloat16",
         "batch": 1, "seq": 8192, "causal": True},
        # A chat-sized prompt of no round length through the GPU-resident cache.
        {"name": "llama-prompt-1999-bf16", "kind": "prompt", "model": "llama3.2-3b", "dtype": "bfloat16",
         "seq": 1999, "max_seq": 4096},
        # The largest decode: 64 long sequences, 2.9 GB of cache read for a token.
        {"name": "llama-decode-bf16", "kind": "decode", "model": "llama3.2-3b", "dtype": "bfloat16", "batch": 64,
         "max_ctx": 16384, "lo": 4096, "hi": 16383, "lens": 4},
        # A prompt's whole layer in the reference models' own type.
        {"name": "smollm2-360m-layer-1023-fp32", "kind": "layer", "model": "smollm2-360m", "dtype": "float32",
         "seq": 1023, "max_seq": 2048},
        # The MLP of a 2048-token prompt: most of a prompt's operations.
        {"name": "llama-mlp-2048-bf16", "kind": "mlp", "model": "llama3.2-3b", "dtype": "bfloat16", "rows": 2048},
        # The MLP of a decode step of 64 sequences: weights read for a few rows.
        {"name": "llama-mlp-64-bf16", "kind": "mlp", "model": "llama3.2-3b", "dtype": "bfloat16", "rows": 64},
        # A generate loop's step at batch 1: norms, projections, cache, head, one after another.
        {"name": "smollm2-360m-token-fp32", "kind": "token", "model": "smollm2-360m", "dtype": "float32",
         "layers": 8, "ctx": 1000, "max_seq": 2048, "vocab": 49152},
        # Sampling for a batch of sequences, top-k at Llama-3.2's vocabulary.
        {"name": "sample-64-top50-fp32", "kind": "sample", "dtype": "float32", "rows": 64, "vocab": 128256,
         "top_k": 50, "temperature": 0.8},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gqa", "prefill", "prompt", "decode", "mlp", "layer", "token", "sample"])
    model = rng.choice(sorted(HEADS))
    dtype = rng.choice(["float32", "float16", "bfloat16", "bfloat16"])
    if kind == "gqa":
        return {"kind": kind, "model": model, "dtype": dtype, "seq": _log(rng, 16, 1024)}
    if kind == "prefill":
        top = 2048 if dtype == "float32" else 6000
        seq = _log(rng, 64, top)
        batch = _log(rng, 1, max(1, min(8, top // seq)))
        return {"kind": kind, "model": model, "dtype": dtype, "batch": batch, "seq": seq,
                "causal": rng.random() < 0.8}
    if kind == "prompt":
        model = rng.choice(sorted(THETA))
        seq = _log(rng, 32, 1500 if dtype == "float32" else 4000)
        return {"kind": kind, "model": model, "dtype": dtype, "seq": seq, "max_seq": 4096}
    if kind == "decode":
        max_ctx = _log(rng, 256, 8192)
        lo = rng.randint(1, max_ctx // 2)
        return {"kind": kind, "model": model, "dtype": dtype, "batch": _log(rng, 1, 48), "max_ctx": max_ctx,
                "lo": lo, "hi": rng.randint(lo, max_ctx - 1), "lens": rng.randint(0, 1 << 20)}
    model = rng.choice(sorted(WIDTH))
    top = 2000 if dtype != "float32" else 1500 if model == "smollm2-360m" else 300
    if kind == "mlp":
        return {"kind": kind, "model": model, "dtype": dtype, "rows": _log(rng, 1, top)}
    if kind == "layer":
        return {"kind": kind, "model": model, "dtype": dtype, "seq": _log(rng, 16, min(top, 1500)), "max_seq": 2048}
    if kind == "token":
        return {"kind": kind, "model": model, "dtype": dtype, "layers": rng.randint(1, 4),
                "ctx": _log(rng, 16, 2000), "max_seq": 2048, "vocab": rng.choice([49152, 32000])}
    return {"kind": kind, "dtype": dtype, "rows": _log(rng, 1, 64), "vocab": _log(rng, 8000, 128256),
            "top_k": rng.choice([0, 1, 20, 50, 100]), "temperature": rng.choice([0.0, 0.6, 0.8, 1.0])}


# ---- a torch tensor and the framework's handle on the same memory ----------

def _dev(t, dtype):
    """The framework's handle on a torch tensor's memory (the tensor stays the owner)."""
    d = gpu.DeviceTensor(ctypes.c_void_p(t.data_ptr()), t.shape, STORE[dtype], t.numel() * t.element_size(),
                         defer_free=False)
    d.owner = t
    return d


class _Shown:
    """A DeviceTensor's memory as an array other programs can look at."""

    def __init__(self, d):
        self.d = d
        kind = {2: "<f2", 4: "<f4"}[d.dtype.itemsize]
        if gpu.dtype_name(d.dtype) == "bfloat16":
            kind = "<i2"
        self.__cuda_array_interface__ = {"shape": d.shape, "typestr": kind, "data": (d.data_ptr(), False),
                                         "strides": None, "version": 2}


def _torch(d):
    """A torch view of a DeviceTensor's memory; it keeps the DeviceTensor."""
    t = torch.as_tensor(_Shown(d), device="cuda")
    return t.view(torch.bfloat16) if gpu.dtype_name(d.dtype) == "bfloat16" else t


class _Make:
    """Seeded inputs on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))
        self.dtype = dtype

    def normal(self, *shape, scale=1.0, mean=0.0):
        if math.prod(shape) > 1 << 28:  # large caches: made in their own type, with no 32-bit copy
            return torch.empty(shape, dtype=TORCH[self.dtype], device="cuda").normal_(mean, scale, generator=self.g)
        x = torch.empty(shape, device="cuda").normal_(mean, scale, generator=self.g)
        return x.to(TORCH[self.dtype])

    def empty(self, *shape):
        return torch.zeros(shape, dtype=TORCH[self.dtype], device="cuda")


def _tables(case, rows):
    cos, sin = precompute_cos_sin(rows, HEADS[case["model"]][2], THETA[case["model"]])
    return torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()


def _table_dev(t):
    return _dev(t, "float32")


def _lens(case):
    return np.random.default_rng(case["lens"]).integers(case["lo"], case["hi"], size=case["batch"],
                                                        endpoint=True).astype(np.int32)


def _layer_weights(mk, model):
    H, Hkv, D = HEADS[model]
    E, I = WIDTH[model]
    return {"ln1": mk.normal(E, scale=0.1, mean=1.0), "ln2": mk.normal(E, scale=0.1, mean=1.0),
            "q": mk.normal(E, H * D, scale=E ** -0.5), "k": mk.normal(E, Hkv * D, scale=E ** -0.5),
            "v": mk.normal(E, Hkv * D, scale=E ** -0.5), "o": mk.normal(H * D, E, scale=(H * D) ** -0.5),
            "gate": mk.normal(E, I, scale=E ** -0.5), "up": mk.normal(E, I, scale=E ** -0.5),
            "down": mk.normal(I, E, scale=I ** -0.5)}


def _inputs(case, seed):
    """The case's values as torch tensors, from the seed alone: what both the
    framework and the 64-bit reference read."""
    kind, dtype = case["kind"], case["dtype"]
    mk = _Make(seed, dtype)
    if kind == "sample":
        # logits of a language model: a few high ones over a broad floor
        x = mk.normal(case["rows"], case["vocab"], scale=2.5)
        u = torch.empty(case["rows"], dtype=torch.float64, device="cuda").uniform_(0.0, 1.0, generator=mk.g)
        return {"logits": x, "u": u}
    H, Hkv, D = HEADS[case["model"]] if "model" in case else (0, 0, 0)
    if kind == "gqa":
        S = case["seq"]
        return {"q": mk.normal(H * S, D), "k": mk.normal(Hkv * S, D), "v": mk.normal(Hkv * S, D)}
    if kind == "prefill":
        B, S = case["batch"], case["seq"]
        return {"q": mk.normal(B, H, S, D), "k": mk.normal(B, Hkv, S, D), "v": mk.normal(B, Hkv, S, D)}
    if kind == "prompt":
        S = case["seq"]
        return {"q": mk.normal(S, H * D), "k": mk.normal(S, Hkv * D), "v": mk.normal(S, Hkv * D)}
    if kind == "decode":
        B, C = case["batch"], case["max_ctx"]
        amp = 0.5 if case["model"] == "gpt2" else 1.0
        return {"q": mk.normal(B, H, D, scale=amp), "k": mk.normal(B, Hkv, D, scale=amp),
                "v": mk.normal(B, Hkv, D, scale=amp), "kc": mk.normal(B, Hkv, C, D, scale=amp),
                "vc": mk.normal(B, Hkv, C, D, scale=amp)}
    E, I = WIDTH[case["model"]]
    if kind == "mlp":
        M = case["rows"]
        w = _layer_weights(mk, case["model"])
        return {"a": mk.normal(M, E), "b": mk.normal(M, E), **{n: w[n] for n in ("ln2", "gate", "up", "down")}}
    if kind == "layer":
        return {"h": mk.normal(case["seq"], E), "w": _layer_weights(mk, case["model"])}
    N, C = case["layers"], case["ctx"]
    return {"h": mk.normal(1, E), "w": [_layer_weights(mk, case["model"]) for _ in range(N)],
            "kc": [mk.normal(Hkv, C, D) for _ in range(N)], "vc": [mk.normal(Hkv, C, D) for _ in range(N)],
            "ln": mk.normal(E, scale=0.1, mean=1.0), "head": mk.normal(E, case["vocab"], scale=E ** -0.5)}


def prepare(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    x = _inputs(case, seed)
    mk = _Make(0, dtype)
    s = {"case": case, "x": x}
    H, Hkv, D = HEADS[case["model"]] if "model" in case else (0, 0, 0)

    def dev(t):
        return _dev(t, dtype)

    def buf(*shape):
        return dev(mk.empty(*shape))

    if kind == "sample":
        tok = torch.zeros(case["rows"], dtype=torch.int32, device="cuda")
        s.update(logits=dev(x["logits"]), tok=tok,
                 u=gpu.DeviceTensor(ctypes.c_void_p(x["u"].data_ptr()), (case["rows"],), np.float64,
                                    8 * case["rows"], defer_free=False),
                 out=gpu.DeviceTensor(ctypes.c_void_p(tok.data_ptr()), (case["rows"],), np.int32,
                                      4 * case["rows"], defer_free=False))
    elif kind == "gqa":
        s.update({n: dev(x[n]) for n in "qkv"})
    elif kind == "prefill":
        s.update({n: dev(x[n]) for n in "qkv"}, out=buf(*x["q"].shape))
    elif kind == "prompt":
        cos, sin = _tables(case, case["max_seq"])
        s.update({n: dev(x[n]) for n in "qkv"}, cos=_table_dev(cos), sin=_table_dev(sin),
                 cache=GpuKVCache(1, H, Hkv, D, max_seq=case["max_seq"], dtype=STORE[dtype]))
    elif kind == "decode":
        s.update({n: dev(x[n]) for n in ("q", "k", "v", "kc", "vc")}, out=buf(*x["q"].shape),
                 cos=None, sin=None, ws=decode_workspace(case["batch"], H, Hkv, case["max_ctx"], D))
        lens = torch.from_numpy(_lens(case)).cuda()
        s.update(lens_t=lens, lens=gpu.DeviceTensor(ctypes.c_void_p(lens.data_ptr()), (case["batch"],), np.int32,
                                                    4 * case["batch"], defer_free=False))
        if case["model"] in THETA:
            cos, sin = _tables(case, case["max_ctx"])
            s.update(cos=_table_dev(cos), sin=_table_dev(sin))
    elif kind == "mlp":
        M, (E, I) = case["rows"], WIDTH[case["model"]]
        s.update({n: dev(t) for n, t in x.items()}, h=buf(M, E), n=buf(M, E), g=buf(M, I), u=buf(M, I),
                 act=buf(M, I), d=buf(M, E), out=buf(M, E))
    elif kind in ("layer", "token"):
        M, (E, I) = case.get("seq", 1), WIDTH[case["model"]]
        cos, sin = _tables(case, case["max_seq"])
        w = [x["w"]] if kind == "layer" else x["w"]
        s.update(cos=_table_dev(cos), sin=_table_dev(sin), h=dev(x["h"]),
                 w=[{n: dev(t) for n, t in lw.items()} for lw in w],
                 cache=GpuKVCache(len(w), H, Hkv, D, max_seq=case["max_seq"], dtype=STORE[dtype]),
                 q=buf(M, H * D), k=buf(M, Hkv * D), v=buf(M, Hkv * D), n1=buf(M, E), o=buf(M, E), h1=buf(M, E),
                 n2=buf(M, E), g=buf(M, I), u=buf(M, I), act=buf(M, I), d=buf(M, E),
                 outs=[buf(M, E) for _ in range(2)])
        if kind == "token":
            s.update(ln=dev(x["ln"]), head=dev(x["head"]), n=buf(1, E), logits=buf(1, case["vocab"]))
            torch.cuda.synchronize()
            for i, c in enumerate(s["cache"].kv_cache_dev):  # what the tokens before this one left in the cache
                _torch(c["k"])[0, :, :case["ctx"]] = x["kc"][i]
                _torch(c["v"])[0, :, :case["ctx"]] = x["vc"][i]
            torch.cuda.synchronize()
            s["cache"].advance(case["ctx"])
            _model(s)  # one pass fills the workspaces
            gpu.synchronize()
            with gpu.capture() as g:
                _model(s)
            s["graph"] = g
    torch.cuda.synchronize()
    return s


def _layer(s, i, h, out):
    """One decoder layer on the rows of h, as the models run it."""
    w = s["w"][i]
    rms_norm(h, w["ln1"], s["n1"])
    gemm_grouped(s["n1"], [w["q"], w["k"], w["v"]], [s["q"], s["k"], s["v"]])
    att = s["cache"].attention(i, s["q"], s["k"], s["v"], s["cos"], s["sin"])
    gemm(att, w["o"], s["o"])
    add_rms_norm(s["o"], h, s["h1"], w["ln2"], s["n2"])
    gemm_grouped(s["n2"], [w["gate"], w["up"]], [s["g"], s["u"]])
    swiglu(s["g"], s["u"], s["act"])
    gemm(s["act"], w["down"], s["d"])
    return add(s["d"], s["h1"], out)


def _model(s):
    h = s["h"]
    for i in range(len(s["w"])):
        h = _layer(s, i, h, s["outs"][i % 2])
    rms_norm(h, s["ln"], s["n"])
    return gemm(s["n"], s["head"], s["logits"])


def run(s):
    case = s["case"]
    kind = case["kind"]
    H, Hkv, D = HEADS[case["model"]] if "model" in case else (0, 0, 0)
    if kind == "gqa":
        return _torch(attention_gqa(s["q"], s["k"], s["v"], H, Hkv, causal=True))
    if kind == "prefill":
        flash_attention(s["q"], s["k"], s["v"], causal=case["causal"], out=s["out"])
        return s["out"].owner
    if kind == "prompt":
        out = s["cache"].attention(0, s["q"], s["k"], s["v"], s["cos"], s["sin"])
        c = s["cache"].kv_cache_dev[0]
        return {"out": _torch(out), "k_cache": _torch(c["k"]), "v_cache": _torch(c["v"])}
    if kind == "decode":
        decode_step(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["lens"], H, Hkv, s["cos"], s["sin"], out=s["out"],
                    workspace=s["ws"])
        return {"out": s["out"].owner, "k_cache": s["kc"].owner, "v_cache": s["vc"].owner}
    if kind == "mlp":
        add_rms_norm(s["a"], s["b"], s["h"], s["ln2"], s["n"])
        gemm_grouped(s["n"], [s["gate"], s["up"]], [s["g"], s["u"]])
        swiglu(s["g"], s["u"], s["act"])
        gemm(s["act"], s["down"], s["d"])
        add(s["d"], s["h"], s["out"])
        return {"out": s["out"].owner, "act": s["act"].owner, "residual": s["h"].owner}
    if kind == "layer":
        out = _layer(s, 0, s["h"], s["outs"][0])
        c = s["cache"].kv_cache_dev[0]
        return {"out": out.owner, "k_cache": _torch(c["k"]), "v_cache": _torch(c["v"])}
    if kind == "token":
        s["graph"].replay()
        caches = s["cache"].kv_cache_dev
        return {"logits": s["logits"].owner, "hidden": s["n"].owner, "k_cache": [_torch(c["k"]) for c in caches],
                "v_cache": [_torch(c["v"]) for c in caches]}
    sample_rows(s["logits"], case["temperature"], case["top_k"], uniforms=s["u"], out_dev=s["out"])
    return s["tok"]


# ---- what a pass cannot do without -------------------------------------------

def _attn_flops(H, D, pairs):
    return 4.0 * D * H * pairs


def _layer_work(case, rows, e):
    H, Hkv, D = HEADS[case["model"]]
    E, I = WIDTH[case["model"]]
    weights = E * (H * D) * 2 + 2 * E * Hkv * D + 3 * E * I
    return {"bytes": float((weights + 2 * E + 2 * rows * E) * e), "flops": 2.0 * rows * weights}


def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    if kind == "sample":
        return {"bytes": float(case["rows"] * (case["vocab"] * e + 12)), "flops": 0.0}
    H, Hkv, D = HEADS[case["model"]]
    if kind in ("gqa", "prefill", "prompt"):
        S, B = case["seq"], case.get("batch", 1)
        pairs = S * (S + 1) / 2 if case.get("causal", True) else S * S
        move = 2 * H + 2 * Hkv + (2 * Hkv if kind == "prompt" else 0)  # a prompt writes its cache rows too
        return {"bytes": float(B * S * D * e * move), "flops": _attn_flops(H, D, B * pairs)}
    if kind == "decode":
        n = int(_lens(case).astype(np.int64).sum())  # cached rows read; the new one is read and written
        B = case["batch"]
        return {"bytes": float((2 * Hkv * n + B * (2 * H + 4 * Hkv)) * D * e), "flops": _attn_flops(H, D, n + B)}
    E, I = WIDTH[case["model"]]
    if kind == "mlp":
        M = case["rows"]
        return {"bytes": float((3 * E * I + E + 3 * M * E) * e), "flops": 6.0 * M * E * I}
    if kind == "layer":
        S = case["seq"]
        w = _layer_work(case, S, e)
        return {"bytes": w["bytes"] + 2.0 * S * Hkv * D * e, "flops": w["flops"] + _attn_flops(H, D, S * (S + 1) / 2)}
    w = _layer_work(case, 1, e)
    N, V, C = case["layers"], case["vocab"], case["ctx"] + 1
    return {"bytes": N * (w["bytes"] + 2.0 * Hkv * C * D * e) + float((E * V + V + E) * e),
            "flops": N * (w["flops"] + _attn_flops(H, D, C)) + 2.0 * E * V}


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "sample":
        return "exact"
    return {"rel": TOLERANCE[kind][dtype]}


# About four times the error against 64 bits, measured: attention 2e-7 in
# float32, 2.2e-4 to 3e-4 in float16, 2.5e-3 to 3.3e-3 in bfloat16 (it rounds
# its probabilities and its output once); the blocks round every intermediate
# (4e-7, 6e-4, 4.7e-3), and a whole model's layers add up.
TOLERANCE = {
    "gqa": {"float32": 1e-6, "float16": 1.5e-3, "bfloat16": 1.2e-2},
    "prefill": {"float32": 1e-6, "float16": 1.5e-3, "bfloat16": 1.2e-2},
    "prompt": {"float32": 1e-6, "float16": 1.5e-3, "bfloat16": 1.2e-2},
    "decode": {"float32": 1e-6, "float16": 1.5e-3, "bfloat16": 1.2e-2},
    "mlp": {"float32": 1.6e-6, "float16": 2.5e-3, "bfloat16": 1.9e-2},
    "layer": {"float32": 1.6e-6, "float16": 2.5e-3, "bfloat16": 1.9e-2},
    "token": {"float32": 2e-6, "float16": 3e-3, "bfloat16": 2.4e-2},
}


# ---- the same in 64 bits --------------------------------------------------------

def _rope64(x, cos, sin, pos):
    """x (..., rows, D) rotated at positions pos (rows,): element i with i + D/2."""
    c, s = cos[pos].double(), sin[pos].double()
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend64(q, k, v, causal):
    """q (H, Sq, D), k / v (Hkv, Sk, D), one head at a time, rows in blocks."""
    H, Sq, D = q.shape
    group = H // k.shape[0]
    Sk = k.shape[1]
    out = torch.empty_like(q)
    keys = torch.arange(Sk, device=q.device)
    for h in range(H):
        kh, vh = k[h // group], v[h // group]
        for r in range(0, Sq, 4096):
            n = min(4096, Sq - r)
            s = (q[h, r:r + n] @ kh.T) / math.sqrt(D)
            if causal:
                s.masked_fill_(keys[None, :] > torch.arange(r, r + n, device=q.device)[:, None] + (Sk - Sq),
                               float("-inf"))
            out[h, r:r + n] = torch.softmax(s, -1) @ vh
    return out


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _mlp64(n, gate, up, down):
    act = torch.nn.functional.silu(n @ gate.double()) * (n @ up.double())
    return act, act @ down.double()


def _layer64(case, h, w, cos, sin, prev_k=None, prev_v=None):
    """h (rows, E) -> the layer's output and its K and V rows (Hkv, ctx, D)."""
    H, Hkv, D = HEADS[case["model"]]
    M = h.shape[0]
    n = _norm64(h, w["ln1"].double())
    q, k, v = ((n @ w[p].double()).view(M, -1, D).transpose(0, 1) for p in "qkv")
    at = 0 if prev_k is None else prev_k.shape[1]
    pos = torch.arange(at, at + M, device=h.device)
    q, k = _rope64(q, cos, sin, pos), _rope64(k, cos, sin, pos)
    if prev_k is not None:
        k, v = torch.cat([prev_k.double(), k], 1), torch.cat([prev_v.double(), v], 1)
    att = _attend64(q.contiguous(), k.contiguous(), v.contiguous(), True).transpose(0, 1).reshape(M, H * D)
    h1 = att @ w["o"].double() + h
    return _mlp64(_norm64(h1, w["ln2"].double()), w["gate"], w["up"], w["down"])[1] + h1, k, v


def _cache64(rows, max_seq):
    c = torch.zeros(1, rows.shape[0], max_seq, rows.shape[2], dtype=torch.float64, device=rows.device)
    c[0, :, :rows.shape[1]] = rows
    return c


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # whole numbers
    x = _inputs(case, seed)
    H, Hkv, D = HEADS[case["model"]]
    if kind == "gqa":
        q, k, v = (x[n].double().view(-1, case["seq"], D) for n in "qkv")
        return _attend64(q, k, v, True).reshape(-1, D)
    if kind == "prefill":
        return torch.stack([_attend64(x["q"][b].double(), x["k"][b].double(), x["v"][b].double(), case["causal"])
                            for b in range(case["batch"])])
    if kind == "prompt":
        S = case["seq"]
        cos, sin = _tables(case, case["max_seq"])
        q, k, v = (x[n].double().view(S, -1, D).transpose(0, 1).contiguous() for n in "qkv")
        pos = torch.arange(S, device="cuda")
        q, k = _rope64(q, cos, sin, pos), _rope64(k, cos, sin, pos)
        out = _attend64(q, k, v, True).transpose(0, 1).reshape(S, H * D)
        return {"out": out, "k_cache": _cache64(k, case["max_seq"]), "v_cache": _cache64(v, case["max_seq"])}
    if kind == "decode":
        lens = _lens(case)
        cos, sin = _tables(case, case["max_ctx"]) if case["model"] in THETA else (None, None)
        out = torch.empty(case["batch"], H, D, dtype=torch.float64, device="cuda")
        new = x["k"].double()
        for b, n in enumerate(int(v) for v in lens):
            q, k, v = x["q"][b].double(), x["k"][b].double(), x["v"][b].double()
            if cos is not None:
                pos = torch.tensor([n], device="cuda")
                q, k = _rope64(q[:, None], cos, sin, pos)[:, 0], _rope64(k[:, None], cos, sin, pos)[:, 0]
            new[b] = k
            K = torch.cat([x["kc"][b, :, :n].double(), k[:, None]], 1)
            V = torch.cat([x["vc"][b, :, :n].double(), v[:, None]], 1)
            s = torch.softmax(torch.matmul(q.view(Hkv, H // Hkv, D), K.transpose(1, 2).contiguous()) / math.sqrt(D), -1)
            out[b] = torch.matmul(s, V).view(H, D)
        if x["kc"].numel() > 1 << 28:
            return {"out": out, "k_cache": None, "v_cache": None}
        kc, vc = x["kc"].double(), x["vc"].double()
        for b, n in enumerate(int(v) for v in lens):
            kc[b, :, n], vc[b, :, n] = new[b], x["v"][b].double()
        return {"out": out, "k_cache": kc, "v_cache": vc}
    if kind == "mlp":
        h = x["a"].double() + x["b"].double()
        act, d = _mlp64(_norm64(h, x["ln2"].double()), x["gate"], x["up"], x["down"])
        return {"out": d + h, "act": act, "residual": h}
    cos, sin = _tables(case, case["max_seq"])
    if kind == "layer":
        out, k, v = _layer64(case, x["h"].double(), x["w"], cos, sin)
        return {"out": out, "k_cache": _cache64(k, case["max_seq"]), "v_cache": _cache64(v, case["max_seq"])}
    h = x["h"].double()
    caches = {"k_cache": [], "v_cache": []}
    for w, kc, vc in zip(x["w"], x["kc"], x["vc"]):
        h, k, v = _layer64(case, h, w, cos, sin, kc, vc)
        caches["k_cache"].append(_cache64(k, case["max_seq"]))
        caches["v_cache"].append(_cache64(v, case["max_seq"]))
    n = _norm64(h, x["ln"].double())
    return {"logits": n @ x["head"].double(), "hidden": n, **caches}
