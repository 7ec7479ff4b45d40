"""What a user of this framework has it do on an MI355X, as cases that can be timed.

A case is a dict of plain values.  listed() names them, draw() gives more of
the same ranges, prepare() makes what a program holds before the call (inputs,
weights, caches, a loaded model, the argument lists of its calls), run() is one
pass through the C ABI, work() the bytes and operations one pass cannot do
without, exact() the same outputs in 64 bits in plain torch, and tolerance()
how far another correct implementation of the same precision may be from this
one.  What each kind of case stands for is said at its listed case.
"""
import ctypes
import glob
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = glob.glob(os.path.join(glob.escape(ROOT), "*_amd"))[0]
if PKG not in sys.path:
    sys.path.insert(0, PKG)
import fence_model  # noqa: E402
import fence_ops as F  # noqa: E402
import gguf_writer  # noqa: E402

NEOX, INTERLEAVED = F.ROPE_NEOX, F.ROPE_INTERLEAVED
EPS = 1e-6
MAX_CTX = 4096


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # A decode step's fused single-row ops at Llama-3-8B size, launch by launch (embed, norm, RoPE, the
        # softmax of 32 heads' scores, norm, SwiGLU): six small launches, where latency is all there is.
        {"name": "token_ops_llama3_8b", "kind": "token_ops", "embed": 4096, "ff": 14336, "heads": 32, "kv_heads": 8,
         "head_dim": 128, "pos": 2915, "vocab": 128256},
        # Prefill of a short prompt: its rows out of the Q8_0 embedding table.
        {"name": "embed_512x4096", "kind": "embed", "tokens": 512, "embed": 4096, "vocab": 128256, "norm": False},
        # Prefill of a large batch: rows gathered and normalised in one pass; ids as a text has them (Zipf).
        {"name": "embed_norm_8192x5120", "kind": "embed", "tokens": 8192, "embed": 5120, "vocab": 151936, "norm": True},
        # Prefill: per-head norm and RoPE of q and k of one layer.
        {"name": "qk_norm_rope_4096", "kind": "rope", "tokens": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "norm": "head", "style": NEOX, "pos": 0},
        # Prefill: a layer boundary on an odd number of tokens (residual add, norm, binary16 for the next GEMM).
        {"name": "residual_norm_2047x4096", "kind": "residual_norm", "tokens": 2047, "embed": 4096},
        # Prefill: causal attention scores of 32 heads.
        {"name": "softmax_causal_32x2048", "kind": "softmax", "heads": 32, "queries": 2048, "keys": 2048},
        # Prefill: the FFN activation of a large batch, the most bytes of all.
        {"name": "swiglu_8192x14336", "kind": "swiglu", "tokens": 8192, "ff": 14336, "half": False},
        # Decode: the attention half of four Qwen3-4B layers at a long context (norm + q/k/v, attention with
        # QK-norm, RoPE and the KV store, o projection).  Every layer has weights and caches of its own, so
        # they come from HBM as they do in a model, and an input of its own, so rounding does not add up.
        {"name": "attn_qwen3_4b_ctx2916", "kind": "attn", "layers": 4, "embed": 2560, "heads": 32, "kv_heads": 8,
         "pos": 2915, "qk_norm": True},
        # Decode: the FFN half of four Qwen3-4B layers (norm + gate/up + SwiGLU, down projection).
        {"name": "mlp_qwen3_4b", "kind": "mlp", "layers": 4, "embed": 2560, "ff": 9728},
        # Decode: the same of two Llama-3-8B layers, with longer rows.
        {"name": "mlp_llama3_8b", "kind": "mlp", "layers": 2, "embed": 4096, "ff": 14336},
        # Decode: the LM head of Llama-3-8B.
        {"name": "lm_head_128256x4096", "kind": "lm_head", "vocab": 128256, "embed": 4096},
        # Decode: one whole step of a Qwen3-4B-shaped model from a GGUF file, at a long context.
        {"name": "model_qwen3_4b_pos2915", "kind": "model", "layers": 36, "embed": 2560, "ff": 9728, "heads": 32,
         "kv_heads": 8, "vocab": 151936, "pos": 2915, "tokens": 1},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["token_ops", "embed", "rope", "residual_norm", "softmax", "swiglu", "attn", "attn", "mlp", "mlp",
                       "lm_head", "model"])
    heads = rng.choice([(32, 8), (32, 8), (16, 8), (40, 8), (64, 8), (14, 2), (16, 16), (6, 2)])
    if kind == "token_ops":
        return {"kind": kind, "embed": _log(rng, 512, 5120, 32), "ff": _log(rng, 1024, 17408, 4), "heads": heads[0],
                "kv_heads": heads[1], "head_dim": rng.choice([128, 128, 64]), "pos": rng.randrange(0, MAX_CTX),
                "vocab": 32000}
    if kind == "embed":
        tokens, embed = _log(rng, 1, 8192), _log(rng, 512, 5120, 32)
        return {"kind": kind, "tokens": tokens, "embed": embed, "vocab": 65536, "norm": rng.random() < 0.5}
    if kind == "rope":
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "heads": heads[0], "kv_heads": heads[1],
                "head_dim": rng.choice([128, 128, 128, 64, 96]), "norm": rng.choice(["none", "head", "row"]),
                "style": rng.choice([NEOX, INTERLEAVED]), "pos": rng.randrange(0, 4096)}
    if kind == "residual_norm":
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "embed": _log(rng, 512, 5120, rng.choice([1, 4, 256]))}
    if kind == "softmax":
        queries = _log(rng, 1, 2048)
        return {"kind": kind, "heads": rng.choice([6, 14, 16, 32]), "queries": queries,
                "keys": max(queries, _log(rng, 64, 4096, rng.choice([1, 4, 64])) if queries < 1024 else queries)}
    if kind == "swiglu":
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "ff": _log(rng, 512, 14336, rng.choice([1, 4, 256])),
                "half": rng.random() < 0.5}
    if kind == "attn":
        return {"kind": kind, "layers": rng.randrange(1, 5), "embed": _log(rng, 512, 5120, 256), "heads": heads[0],
                "kv_heads": heads[1], "pos": min(MAX_CTX - 1, _log(rng, 1, MAX_CTX) - 1), "qk_norm": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "layers": rng.randrange(1, 4), "embed": _log(rng, 512, 5120, 256),
                "ff": _log(rng, 1024, 17408, 256)}
    if kind == "lm_head":
        return {"kind": kind, "vocab": _log(rng, 8192, 131072), "embed": _log(rng, 512, 5120, rng.choice([32, 256]))}
    tokens = rng.choice([1, 1, 2, 4])
    return {"kind": "model", "layers": rng.randrange(1, 13), "embed": _log(rng, 512, 4096, 256),
            "ff": _log(rng, 1024, 12288, 256), "heads": heads[0], "kv_heads": heads[1], "vocab": _log(rng, 8192, 131072),
            "pos": min(MAX_CTX - 8, _log(rng, 1, MAX_CTX) - 1), "tokens": tokens}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 11)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * std


def _norm_weight(g, n):
    return 1 + 0.1 * _randn(g, n)


def _q6k(g, rows, k):
    """[rows, k/256, 210] Q6_K blocks: weights of standard deviation about 0.02, sub-block scales of either
    sign from 32 to 127, as a quantiser that scales the largest to 127 leaves them, and d around 1.3e-5 (a
    subnormal binary16, which such weights have)."""
    nb = k // 256
    w = torch.randint(0, 256, (rows, nb, 210), dtype=torch.uint8, device="cuda", generator=g)
    sc = torch.randint(32, 128, (rows, nb, 16), dtype=torch.int16, device="cuda", generator=g)
    sign = w[:, :, 192:208].to(torch.int16) & 1
    w[:, :, 192:208] = torch.where(sign == 1, -sc, sc).to(torch.int8).view(torch.uint8)
    d = (1.3e-5 * (0.5 + torch.rand(rows, nb, 1, device="cuda", generator=g))).half()
    w[:, :, 208:210] = d.view(torch.uint8).view(rows, nb, 2)
    return w


def _q8_0(g, rows, k):
    """[rows, k/32, 34] Q8_0 blocks: values of standard deviation about 0.02."""
    nb = k // 32
    w = torch.randint(0, 256, (rows, nb, 34), dtype=torch.uint8, device="cuda", generator=g)
    d = (2.7e-4 * (0.5 + torch.rand(rows, nb, 1, device="cuda", generator=g))).half()
    w[:, :, 0:2] = d.view(torch.uint8).view(rows, nb, 2)
    q = w[:, :, 2:]
    q[q == 128] = 129  # a quantiser gives -127 .. 127
    return w


def _ids(g, tokens, vocab):
    """Zipf(1.1) token ids, as a text has them."""
    cdf = torch.cumsum(torch.arange(1, vocab + 1, dtype=torch.float64, device="cuda") ** -1.1, 0)
    u = torch.rand(tokens, dtype=torch.float64, device="cuda", generator=g) * cdf[-1]
    return torch.clamp(torch.searchsorted(cdf, u), max=vocab - 1).to(torch.int32)


def _scores(g, heads, queries, keys):
    """Scores [heads, queries, keys]; the keys a query does not see are at -inf, as a mask leaves them."""
    s = _randn(g, heads, queries, keys, std=3.0 / 128 ** 0.5)
    mask = torch.ones(queries, keys, dtype=torch.bool, device="cuda").triu_(1 + keys - queries)
    return s.masked_fill_(mask, float("-inf"))


def _inputs(case, seed):
    """The case's inputs as a dict of device tensors, from the seed alone."""
    g, c, kind = _gen(seed), case, case["kind"]
    if kind == "token_ops":
        hd = c["head_dim"]
        return {"table": _q8_0(g, c["vocab"], c["embed"]), "w1": _norm_weight(g, c["embed"]),
                "w2": _norm_weight(g, c["embed"]), "q": _randn(g, c["heads"], hd), "k": _randn(g, c["kv_heads"], hd),
                "scores": _randn(g, c["heads"], MAX_CTX, std=3.0 / 128 ** 0.5), "gate": _randn(g, c["ff"]),
                "up": _randn(g, c["ff"]), "token": 17 + int(seed) % (c["vocab"] - 17)}
    if kind == "embed":
        return {"table": _q8_0(g, c["vocab"], c["embed"]), "ids": _ids(g, c["tokens"], c["vocab"]),
                "w": _norm_weight(g, c["embed"])}
    if kind == "rope":
        t, hd = c["tokens"], c["head_dim"]
        x = {"q": _randn(g, t, c["heads"], hd), "k": _randn(g, t, c["kv_heads"], hd)}
        if c["norm"] == "head":
            x["wq"], x["wk"] = _norm_weight(g, hd), _norm_weight(g, hd)
        elif c["norm"] == "row":
            x["wq"] = _norm_weight(g, c["heads"] * hd)
        return x
    if kind == "residual_norm":
        t, e = c["tokens"], c["embed"]
        return {"hidden": _randn(g, t, e), "residual": _randn(g, t, e), "w": _norm_weight(g, e)}
    if kind == "softmax":
        return {"x": _scores(g, c["heads"], c["queries"], c["keys"])}
    if kind == "swiglu":
        return {"gate": _randn(g, c["tokens"], c["ff"]), "up": _randn(g, c["tokens"], c["ff"])}
    if kind == "lm_head":
        return {"table": _q8_0(g, c["vocab"], c["embed"]), "x": _randn(g, c["embed"])}
    layers, e = c["layers"], c["embed"]
    if kind == "mlp":
        return {"hidden": _randn(g, layers, e), "residual": _randn(g, layers, e),
                "w": [_norm_weight(g, e) for _ in range(layers)],
                "gate": [_q6k(g, c["ff"], e) for _ in range(layers)], "up": [_q6k(g, c["ff"], e) for _ in range(layers)],
                "down": [_q6k(g, e, c["ff"]) for _ in range(layers)]}
    if kind == "attn":
        q, kv = c["heads"] * 128, c["kv_heads"] * 128
        cache = (layers, MAX_CTX, c["kv_heads"], 128)
        return {"hidden": _randn(g, layers, e), "residual": _randn(g, layers, e),
                "w": [_norm_weight(g, e) for _ in range(layers)],
                "wq": [_q6k(g, q, e) for _ in range(layers)], "wk": [_q6k(g, kv, e) for _ in range(layers)],
                "wv": [_q6k(g, kv, e) for _ in range(layers)], "wo": [_q6k(g, e, q) for _ in range(layers)],
                "nq": [_norm_weight(g, 128) for _ in range(layers)], "nk": [_norm_weight(g, 128) for _ in range(layers)],
                "kc": _randn(g, *cache).half(), "vc": _randn(g, *cache).half()}
    # model: the tensors of its file, under their names there, and the KV caches' contents
    q, kv, ff = c["heads"] * 128, c["kv_heads"] * 128, c["ff"]
    t = {"token_embd.weight": _q8_0(g, c["vocab"], e), "output_norm.weight": _norm_weight(g, e)}
    for l in range(layers):
        p = "blk.%d." % l
        t[p + "attn_norm.weight"] = _norm_weight(g, e)
        t[p + "attn_q.weight"], t[p + "attn_k.weight"] = _q6k(g, q, e), _q6k(g, kv, e)
        t[p + "attn_v.weight"] = _q6k(g, kv, e)
        t[p + "attn_q_norm.weight"], t[p + "attn_k_norm.weight"] = _norm_weight(g, 128), _norm_weight(g, 128)
        t[p + "attn_output.weight"] = _q6k(g, e, q)
        t[p + "ffn_norm.weight"] = _norm_weight(g, e)
        t[p + "ffn_gate.weight"], t[p + "ffn_up.weight"] = _q6k(g, ff, e), _q6k(g, ff, e)
        t[p + "ffn_down.weight"] = _q6k(g, e, ff)
    # one pool of rows serves every layer's caches, from another row on
    pool = _randn(g, 2, c["pos"] + 64 * layers + 8, c["kv_heads"], 128).half()
    tokens = [(97 * int(seed) + 31 * i + 5) % c["vocab"] for i in range(c["tokens"])]
    return {"tensors": t, "pool": pool, "tokens": tokens}


# ------------------------------------------------------------------ a pass

class _DeviceArray:
    """Device memory of the library's as something torch can view; the view keeps its owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_DeviceArray(owner, ptr, shape, typestr), device="cuda")


_streams = []


def _model_stream():
    """The one stream that this process's models decode on, as a program serving one request after another has."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0].cuda_stream


def _p(t):
    return ctypes.c_void_p(None if t is None else t.data_ptr())


def _arr(ctype, values):
    return (ctype * len(values))(*values)


def prepare(case, seed):
    c, kind, x = case, case["kind"], _inputs(case, seed)
    lib = F.lib()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    f32 = dict(dtype=torch.float32, device="cuda")
    f16 = dict(dtype=torch.float16, device="cuda")
    calls, out = [], {}
    if kind == "token_ops":
        e, ff, heads, hd = c["embed"], c["ff"], c["heads"], c["head_dim"]
        out = {"hidden": torch.empty(e, **f32), "normed1": torch.empty(e, **f32), "normed2": torch.empty(e, **f32),
               "q": x["q"], "k": x["k"], "scores": x["scores"], "act": torch.empty(ff, **f32)}
        calls = [
            (lib.fence_embed_q8_0, (_p(out["hidden"]), _p(x["table"]), x["token"], e, s)),
            (lib.fence_rms_norm, (_p(out["normed1"]), _p(out["hidden"]), _p(x["w1"]), e, EPS, s)),
            (lib.fence_rope, (_p(x["q"]), _p(x["k"]), 1, heads, c["kv_heads"], hd, None, c["pos"], 5e5, INTERLEAVED, s)),
            (lib.fence_softmax_rows, (_p(x["scores"]), heads, c["pos"] + 1, MAX_CTX, s)),
            (lib.fence_rms_norm, (_p(out["normed2"]), _p(out["hidden"]), _p(x["w2"]), e, EPS, s)),
            (lib.fence_silu_elementwise_mul, (_p(out["act"]), _p(x["gate"]), _p(x["up"]), ff, s))]
    elif kind == "embed":
        out = {"out": torch.empty(c["tokens"], c["embed"], **f32)}
        args = (_p(out["out"]), _p(x["table"]), c["vocab"], _p(x["ids"]), c["tokens"], c["embed"])
        calls = [(lib.fence_embed_q8_0_gather_rms_norm, args + (_p(x["w"]), EPS, s)) if c["norm"]
                 else (lib.fence_embed_q8_0_gather, args + (s,))]
    elif kind == "rope":
        tail = (c["tokens"], c["heads"], c["kv_heads"], c["head_dim"])
        pos = (None, c["pos"], 1e6, c["style"], s)
        if c["norm"] == "head":
            calls = [(lib.fence_qk_norm_rope, (_p(x["q"]), _p(x["k"]), _p(x["wq"]), _p(x["wk"])) + tail + (EPS,) + pos)]
            out = {"q": x["q"], "k": x["k"]}
        elif c["norm"] == "row":
            out = {"q": torch.empty_like(x["q"]), "k": x["k"]}
            calls = [(lib.fence_rms_norm_rope, (_p(out["q"]), _p(x["q"]), _p(x["wq"]), _p(x["k"])) + tail + (EPS,) + pos)]
        else:
            calls = [(lib.fence_rope, (_p(x["q"]), _p(x["k"])) + tail + pos)]
            out = {"q": x["q"], "k": x["k"]}
    elif kind == "residual_norm":
        out = {"hidden": x["hidden"], "x16": torch.empty(c["tokens"], c["embed"], **f16)}
        calls = [(lib.fence_residual_rms_norm_f16, (_p(x["hidden"]), _p(x["residual"]), _p(x["w"]), None, _p(out["x16"]),
                                                    c["tokens"], c["embed"], EPS, s))]
    elif kind == "softmax":
        out = {"x": x["x"]}
        calls = [(lib.fence_softmax_causal, (_p(x["x"]), c["heads"], c["queries"], c["keys"], s))]
    elif kind == "swiglu":
        n = c["tokens"] * c["ff"]
        out = {"act": torch.empty(c["tokens"], c["ff"], **(f16 if c["half"] else f32))}
        calls = [(lib.fence_swiglu_f16, (_p(out["act"]), None, _p(x["gate"]), _p(x["up"]), n, s)) if c["half"]
                 else (lib.fence_swiglu, (_p(out["act"]), _p(x["gate"]), _p(x["up"]), n, s))]
    elif kind == "lm_head":
        out = {"logits": torch.empty(c["vocab"], **f32)}
        calls = [(lib.fence_gemv_q8_0, (_p(x["table"]), _p(x["x"]), _p(out["logits"]), c["vocab"], c["embed"], s))]
    elif kind == "mlp":
        layers, e, ff = c["layers"], c["embed"], c["ff"]
        out = {"hidden": torch.empty(layers, e, **f32), "x16": torch.empty(layers, e, **f16),
               "act16": torch.empty(layers, ff, **f16), "down": torch.empty(layers, e, **f32)}
        for l in range(layers):
            rin = F.rms_input(x["hidden"][l].data_ptr(), x["residual"][l].data_ptr(), out["hidden"][l].data_ptr(),
                              x["w"][l].data_ptr(), out["x16"][l].data_ptr(), EPS)
            calls += [(lib.fence_gemv_q6k_swiglu_rms_f16, (_p(x["gate"][l]), _p(x["up"][l]), ctypes.pointer(rin),
                                                           _p(out["act16"][l]), None, ff, e, s)),
                      (lib.fence_gemv_q6k, (_p(x["down"][l]), _p(out["act16"][l]), _p(out["down"][l]), e, ff, s))]
    elif kind == "attn":
        layers, e, heads, kvh, pos = c["layers"], c["embed"], c["heads"], c["kv_heads"], c["pos"]
        q, kv = heads * 128, kvh * 128
        out = {"hidden": torch.empty(layers, e, **f32), "x16": torch.empty(layers, e, **f16),
               "attn16": torch.empty(layers, q, **f16), "o": torch.empty(layers, e, **f32),
               "k_row": x["kc"][:, pos], "v_row": x["vc"][:, pos]}
        x["qkv"] = torch.empty(layers, q + 2 * kv, **f32)
        x["scratch"] = torch.empty(4 * heads * MAX_CTX, **f32)
        x["arrive"] = torch.zeros(heads * F.ARRIVE_WORDS_PER_HEAD, dtype=torch.int32, device="cuda")
        for l in range(layers):
            rin = F.rms_input(x["hidden"][l].data_ptr(), x["residual"][l].data_ptr(), out["hidden"][l].data_ptr(),
                              x["w"][l].data_ptr(), out["x16"][l].data_ptr(), EPS)
            yq = x["qkv"][l].data_ptr()
            yk, yv = yq + 4 * q, yq + 4 * (q + kv)
            nq, nk = (_p(x["nq"][l]), _p(x["nk"][l])) if c["qk_norm"] else (None, None)
            calls += [
                (lib.fence_gemv_q6k_multi_rms,
                 (3, _arr(ctypes.c_void_p, [x["wq"][l].data_ptr(), x["wk"][l].data_ptr(), x["wv"][l].data_ptr()]),
                  _arr(ctypes.c_void_p, [yq, yk, yv]), None, _arr(ctypes.c_int, [q, kv, kv]), ctypes.pointer(rin), e, s)),
                (lib.fence_gqa_attention_qk_f16_arrive,
                 (None, _p(out["attn16"][l]), ctypes.c_void_p(yq), ctypes.c_void_p(yk), ctypes.c_void_p(yv), nq, nk,
                  _p(x["kc"][l]), _p(x["vc"][l]), 128, heads, kvh, pos, MAX_CTX, EPS, 1e6, NEOX, _p(x["scratch"]),
                  x["scratch"].numel(), _p(x["arrive"]), s)),
                (lib.fence_gemv_q6k, (_p(x["wo"][l]), _p(out["attn16"][l]), _p(out["o"][l]), e, q, s))]
    else:
        return _prepare_model(case, x)
    return {"calls": calls, "out": out, "inputs": x}


def _prepare_model(c, x):
    kinds = {"token_embd.weight": gguf_writer.Q8_0}
    dims = {}
    for n, t in x["tensors"].items():
        if t.dim() == 1:
            kinds[n], dims[n] = gguf_writer.F32, [t.numel()]
        else:
            kinds.setdefault(n, gguf_writer.Q6_K)
            dims[n] = [t.shape[1] * (32 if kinds[n] == gguf_writer.Q8_0 else 256), t.shape[0]]
    u, f, st = gguf_writer.UINT32, gguf_writer.FLOAT32, gguf_writer.STRING
    meta = [("general.architecture", st, "qwen3"), ("qwen3.block_count", u, c["layers"]),
            ("qwen3.embedding_length", u, c["embed"]), ("qwen3.feed_forward_length", u, c["ff"]),
            ("qwen3.attention.head_count", u, c["heads"]), ("qwen3.attention.head_count_kv", u, c["kv_heads"]),
            ("qwen3.attention.key_length", u, 128), ("qwen3.rope.freq_base", f, 1e6),
            ("qwen3.attention.layer_norm_rms_epsilon", f, EPS)]
    fd, path = tempfile.mkstemp(suffix=".gguf", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    os.close(fd)
    try:
        gguf_writer.write_gguf(path, meta, [(n, dims[n], kinds[n], (lambda t=t: t.cpu().numpy().reshape(-1).view(np.uint8)),
                                             t.numel() * t.element_size()) for n, t in x["tensors"].items()])
        x["tensors"] = None
        m = fence_model.Model(path, max_ctx=MAX_CTX, stream=_model_stream())
    finally:
        os.remove(path)
    kv, pos = c["kv_heads"] * 128, c["pos"]
    rows = []
    for l in range(c["layers"]):
        pk, pv = m.kv_cache(l)
        k, v = _view(m, pk, (MAX_CTX, kv), "<f2"), _view(m, pv, (MAX_CTX, kv), "<f2")
        k[:pos] = x["pool"][0, 64 * l:64 * l + pos].view(pos, kv)
        v[:pos] = x["pool"][1, 64 * l:64 * l + pos].view(pos, kv)
        if l in (0, c["layers"] - 1):
            rows += [k[pos:pos + c["tokens"]], v[pos:pos + c["tokens"]]]
    torch.cuda.synchronize()  # the caches are filled before the model's own stream reads them
    return {"model": m, "tokens": x["tokens"], "pos": pos, "vocab": c["vocab"], "rows": rows}


def run(state):
    if "model" in state:
        m, logits = state["model"], None
        for i, t in enumerate(state["tokens"]):
            logits = m.forward(t, state["pos"] + i)
        return {"logits": _view(m, logits, (state["vocab"],), "<f4"), "rows": state["rows"]}
    for fn, args in state["calls"]:
        status = fn(*args)
        if status:
            raise F.FenceError(fn.__name__, status)
    return state["out"]


# ------------------------------------------------------------------ work and tolerance

def _q6k_bytes(rows, k):
    return rows * (k // 256) * 210


def work(case):
    c, kind = case, case["kind"]
    if kind == "token_ops":
        e, ff, hd = c["embed"], c["ff"], c["heads"] * c["head_dim"] + c["kv_heads"] * c["head_dim"]
        n = c["heads"] * (c["pos"] + 1)
        return {"bytes": 34 * e // 32 + 4 * e + 2 * 12 * e + 8 * hd + 8 * n + 12 * ff,
                "flops": 10 * e + 6 * hd + 5 * n + 6 * ff}
    if kind == "embed":
        t, e = c["tokens"], c["embed"]
        p = np.arange(1, c["vocab"] + 1, dtype=np.float64) ** -1.1
        rows = int(np.sum(1 - (1 - p / p.sum()) ** t))  # as many rows are distinct under the Zipf law
        return {"bytes": 4 * t * e + rows * 34 * e // 32 + 4 * t + (4 * e if c["norm"] else 0),
                "flops": t * e * (5 if c["norm"] else 1)}
    if kind == "rope":
        n = c["tokens"] * (c["heads"] + c["kv_heads"]) * c["head_dim"]
        w = {"none": 0, "head": 2 * c["head_dim"], "row": c["heads"] * c["head_dim"]}[c["norm"]]
        return {"bytes": 8 * n + 4 * w, "flops": (3 if c["norm"] == "none" else 7) * n}
    if kind == "residual_norm":
        n = c["tokens"] * c["embed"]
        return {"bytes": 14 * n + 4 * c["embed"], "flops": 5 * n}
    if kind == "softmax":
        h, sq, sk = c["heads"], c["queries"], c["keys"]
        seen = h * (sq * (sk - sq) + sq * (sq + 1) // 2)
        return {"bytes": 4 * seen + 4 * h * sq * sk, "flops": 5 * seen}
    if kind == "swiglu":
        n = c["tokens"] * c["ff"]
        return {"bytes": n * (10 if c["half"] else 12), "flops": 6 * n}
    if kind == "lm_head":
        v, e = c["vocab"], c["embed"]
        return {"bytes": v * (e // 32) * 34 + 4 * e + 4 * v, "flops": 2 * v * e}
    e = c["embed"]
    mlp = attn = mlp_flops = attn_flops = 0
    if kind in ("mlp", "model"):
        ff = c["ff"]
        mlp = 2 * _q6k_bytes(ff, e) + _q6k_bytes(e, ff) + 22 * e + 4 * ff
        mlp_flops = 6 * e * ff
    if kind in ("attn", "model"):
        q, kv, n = c["heads"] * 128, c["kv_heads"] * 128, c["pos"] + 1
        attn = _q6k_bytes(q + 2 * kv, e) + _q6k_bytes(e, q) + 4 * n * kv + 22 * e + 8 * (q + 2 * kv) + 4 * q
        attn_flops = 2 * e * (2 * q + 2 * kv) + 4 * q * n
    total = {"bytes": c["layers"] * (mlp + attn), "flops": c["layers"] * (mlp_flops + attn_flops)}
    if kind == "model":
        v = c["vocab"]
        total["bytes"] = c["tokens"] * (total["bytes"] + v * (e // 32) * 34 + 4 * v)
        total["flops"] = c["tokens"] * (total["flops"] + 2 * v * e)
    return total


def tolerance(case):
    kind = case["kind"]
    if kind == "embed" and not case["norm"]:
        return "exact"  # a binary16 scale times an int8 is exact in fp32
    if kind in ("residual_norm",) or (kind == "swiglu" and case["half"]):
        return {"rel": 2e-5, "max": 4e-3}  # a value beside a binary16 tie may round the other way
    if kind in ("mlp", "attn"):
        return {"rel": 2e-4, "max": 4e-3}  # so may some of the values between two projections
    if kind == "model":
        return {"rel": 1e-2, "max": 6e-2}  # a rounding in one layer travels through all that follow
    return {"rel": 2e-6, "max": 1e-5}


# ------------------------------------------------------------------ the same in 64 bits

def _deq_q8_0(w):
    d = w[..., 0:2].contiguous().view(torch.float16).double()
    q = w[..., 2:].contiguous().view(torch.int8).double()
    return (d * q).reshape(w.shape[0], -1)


def _deq_q6k(w):
    m, nb = w.shape[:2]
    ql = w[:, :, :128].to(torch.int16).view(m, nb, 2, 2, 32)
    qh = w[:, :, 128:192].to(torch.int16).view(m, nb, 2, 32)
    sc = w[:, :, 192:208].contiguous().view(torch.int8).double().view(m, nb, 2, 4, 2, 1)
    d = w[:, :, 208:210].contiguous().view(torch.float16).double().view(m, nb, 1, 1, 1, 1)
    q = torch.stack([(ql[:, :, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, :, 1] >> 4) | (((qh >> 6) & 3) << 4)], 3)
    return ((q.double() - 32).view(m, nb, 2, 4, 2, 16) * sc * d).reshape(m, nb * 256)


def _mv(w, x, deq=_deq_q6k):
    step = max(1, (1 << 25) // (w.shape[1] * 256))
    return torch.cat([deq(w[r:r + step]) @ x for r in range(0, w.shape[0], step)])


def _rms(x, w):
    return w.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rope(x, pos, base, style):
    """x [tokens, heads, hd] at positions pos ..: the angle is the fp32 product of the position and the fp32
    frequency 1 / powf(base, 2p / hd), which is what the op is defined with."""
    t, _, hd = x.shape
    e = (np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)).astype(np.float64)
    freq = (np.float32(1) / np.power(np.float64(np.float32(base)), e).astype(np.float32)).astype(np.float32)
    a = np.arange(pos, pos + t, dtype=np.float32)[:, None] * freq[None, :]
    a = torch.from_numpy(a.astype(np.float64)).to(x.device)
    cos, sin = a.cos()[:, None, :], a.sin()[:, None, :]
    x0, x1 = (x[..., :hd // 2], x[..., hd // 2:]) if style == NEOX else (x[..., 0::2], x[..., 1::2])
    y0, y1 = x0 * cos - x1 * sin, x0 * sin + x1 * cos
    return torch.cat([y0, y1], -1) if style == NEOX else torch.stack([y0, y1], -1).flatten(-2)


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _h(x):
    """Through binary16, where the op is defined to round to it."""
    return x.half().double()


def _attention(q, k, v, kc, vc, pos, nq, nk, heads, kv_heads):
    """One token's attention over the caches' rows 0 .. pos - 1 and its own k and v; all 64-bit but the caches."""
    q, k = q.view(heads, 128), k.view(kv_heads, 128)
    if nq is not None:
        q, k = _rms(q, nq), _rms(k, nk)
    q, k = _rope(q[None], pos, 1e6, NEOX)[0], _h(_rope(k[None], pos, 1e6, NEOX)[0])
    v = _h(v.view(kv_heads, 128))
    keys = torch.cat([kc[:pos].double().view(pos, kv_heads, 128), k[None]])
    vals = torch.cat([vc[:pos].double().view(pos, kv_heads, 128), v[None]])
    qg = q.view(kv_heads, heads // kv_heads, 128)
    s = torch.matmul(qg, keys.permute(1, 2, 0).contiguous()) / math.sqrt(128)
    return torch.matmul(torch.softmax(s, -1), vals.permute(1, 0, 2).contiguous()).reshape(-1), k, v


def exact(case, seed):
    c, kind = case, case["kind"]
    x = _inputs(case, seed)
    if kind == "token_ops":
        hidden = _deq_q8_0(x["table"][x["token"]:x["token"] + 1])[0]
        scores = x["scores"].double()
        n = c["pos"] + 1
        scores[:, :n] = torch.softmax(scores[:, :n], -1)
        return {"hidden": hidden, "normed1": _rms(hidden, x["w1"]), "normed2": _rms(hidden, x["w2"]),
                "q": _rope(x["q"].double()[None], c["pos"], 5e5, INTERLEAVED)[0],
                "k": _rope(x["k"].double()[None], c["pos"], 5e5, INTERLEAVED)[0], "scores": scores,
                "act": _silu_mul(x["gate"].double(), x["up"].double())}
    if kind == "embed":
        rows = _deq_q8_0(x["table"][x["ids"].long()])
        return {"out": _rms(rows, x["w"]) if c["norm"] else rows}
    if kind == "rope":
        q, k = x["q"].double(), x["k"].double()
        if c["norm"] == "head":
            q, k = _rms(q, x["wq"]), _rms(k, x["wk"])
        elif c["norm"] == "row":
            q = _rms(q.flatten(1), x["wq"]).view_as(q)
        return {"q": _rope(q, c["pos"], 1e6, c["style"]), "k": _rope(k, c["pos"], 1e6, c["style"])}
    if kind == "residual_norm":
        hidden = x["hidden"].double() + x["residual"].double()
        return {"hidden": hidden, "x16": _h(_rms(hidden.float().double(), x["w"]))}
    if kind == "softmax":
        return {"x": torch.stack([torch.softmax(h.double(), -1) for h in x["x"]])}
    if kind == "swiglu":
        act = _silu_mul(x["gate"].double(), x["up"].double())
        return {"act": _h(act) if c["half"] else act}
    if kind == "lm_head":
        return {"logits": _mv(x["table"], x["x"].double(), _deq_q8_0)}
    if kind == "mlp":
        out = {"hidden": [], "x16": [], "act16": [], "down": []}
        for l in range(c["layers"]):
            hidden = x["hidden"][l].double() + x["residual"][l].double()
            x16 = _h(_rms(hidden.float().double(), x["w"][l]))
            act = _h(_silu_mul(_mv(x["gate"][l], x16), _mv(x["up"][l], x16)))
            for n, v in (("hidden", hidden), ("x16", x16), ("act16", act), ("down", _mv(x["down"][l], act))):
                out[n].append(v)
        return {n: torch.stack(v) for n, v in out.items()}
    if kind == "attn":
        out = {"hidden": [], "x16": [], "attn16": [], "o": [], "k_row": [], "v_row": []}
        for l in range(c["layers"]):
            hidden = x["hidden"][l].double() + x["residual"][l].double()
            x16 = _h(_rms(hidden.float().double(), x["w"][l]))
            norms = (x["nq"][l], x["nk"][l]) if c["qk_norm"] else (None, None)
            a, k, v = _attention(_mv(x["wq"][l], x16), _mv(x["wk"][l], x16), _mv(x["wv"][l], x16), x["kc"][l], x["vc"][l],
                                 c["pos"], *norms, c["heads"], c["kv_heads"])
            a16 = _h(a)
            for n, v_ in (("hidden", hidden), ("x16", x16), ("attn16", a16), ("o", _mv(x["wo"][l], a16)), ("k_row", k),
                          ("v_row", v)):
                out[n].append(v_)
        return {n: torch.stack(v) for n, v in out.items()}
    return _exact_model(c, x)


def _exact_model(c, x):
    t, layers, pos, kv = x["tensors"], c["layers"], c["pos"], c["kv_heads"] * 128
    kc = [x["pool"][0, 64 * l:64 * l + pos].reshape(pos, kv) for l in range(layers)]
    vc = [x["pool"][1, 64 * l:64 * l + pos].reshape(pos, kv) for l in range(layers)]
    logits = None
    for i, token in enumerate(x["tokens"]):
        hidden = _deq_q8_0(t["token_embd.weight"][token:token + 1])[0]
        for l in range(layers):
            w = lambda n, p="blk.%d." % l: t[p + n + ".weight"]  # noqa: E731
            x16 = _h(_rms(hidden, w("attn_norm")))
            a, k, v = _attention(_mv(w("attn_q"), x16), _mv(w("attn_k"), x16), _mv(w("attn_v"), x16), kc[l], vc[l],
                                 pos + i, w("attn_q_norm"), w("attn_k_norm"), c["heads"], c["kv_heads"])
            kc[l] = torch.cat([kc[l], k.half().view(1, kv)])
            vc[l] = torch.cat([vc[l], v.half().view(1, kv)])
            hidden = hidden + _mv(w("attn_output"), _h(a))
            x16 = _h(_rms(hidden, w("ffn_norm")))
            hidden = hidden + _mv(w("ffn_down"), _h(_silu_mul(_mv(w("ffn_gate"), x16), _mv(w("ffn_up"), x16))))
        logits = _mv(t["token_embd.weight"], _rms(hidden, t["output_norm.weight"]), _deq_q8_0)
    rows = []
    for l in sorted({0, layers - 1}):
        rows += [kc[l][pos:].double(), vc[l][pos:].double()]
    return {"logits": logits, "rows": rows}
