"""The work that is timed: layers and blocks of the models this op surface serves, through its public
entry points (the Python binding and the C ABI it wraps), on one GPU.

Every case is one of these kinds; `listed()` names twelve of them and `draw()` gives others of the same
ranges (1 to 4096 tokens, odd counts among them, projections of 512 to 4304 columns):

  mlp_w8a8     RMSNorm + per-token int8, the gate|up Q8_0 GEMM with its glue, re-quantize, down GEMM
  mlp_f16      RMSNorm, the fp16 gate|up GEMM with its glue, the fp16 down GEMM
  attn_layer   RMSNorm, fused q|k|v GEMM, q/k norm + RoPE + attention on that buffer, output GEMM
  linear_i8    the group-wise int8 projection: activations quantized per row and group, then the product
  linear_f16   one fp16 projection
  vision       the four GEMMs and the bidirectional attention of a vision-tower layer
  attention    masked grouped-query attention of n_q queries on n_kv keys (prefill, chunk or decode)
  moe          the routed expert FFN of a mixture-of-experts layer, bucketed by the call's router choice
  host_linear  a projection on ordinary host arrays (fp16, Q8_0, group-wise int8 or QAT weight)

Device cases run on the library's stream on tensors that stay in HBM, as a program with its activations on
the GPU does; `host_linear` takes and returns numpy arrays, as the reference's callers do.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "burn-rocket_amd"))
import burn_rocket as rk  # noqa: E402

EPS = 1e-6


def listed():
    return [
        # a search query (a dozen tokens) through a 0.6B embedding model's Q8_0 MLP: launches and latency
        dict(name="query_mlp_w8a8", kind="mlp_w8a8", m=12, hidden=1024, inter=3072, glu="silu"),
        # the same query through the model's attention layer, fp16 weights
        dict(name="query_attn_layer", kind="attn_layer", s=24, hidden=1024, h=16, kv=8, d=128),
        # a paragraph through the fp16 MLP
        dict(name="passage_mlp_f16", kind="mlp_f16", m=512, hidden=1024, inter=3072, glu="silu"),
        # a document of 3633 tokens through the attention layer and through the Q8_0 MLP
        dict(name="document_attn_layer", kind="attn_layer", s=3633, hidden=1024, h=16, kv=8, d=128),
        dict(name="document_mlp_w8a8", kind="mlp_w8a8", m=3633, hidden=1024, inter=3072, glu="silu"),
        # a document through a projection packed group-wise (128 values a scale)
        dict(name="document_linear_i8", kind="linear_i8", m=2777, k=1024, n=3072, group=128),
        # one layer of the vision tower on a full page of patches
        dict(name="page_vision", kind="vision", s=2394, hidden=1152, h=16, d=72, mlp=4304),
        # a sliding-window layer of a text encoder with one kv head of 256
        dict(name="window_attention", kind="attention", n_q=2587, n_kv=2587, h=3, kv=1, d=256, mode="window",
             window=512),
        # one generated token against the keys so far
        dict(name="decode_attention", kind="attention", n_q=1, n_kv=4096, h=32, kv=4, d=128, mode="causal", window=-1),
        # the experts of a 30B-A3B layer on a prompt, and on a few sequences that generate
        dict(name="prompt_moe", kind="moe", s=1024, hidden=2048, experts=128, top_k=8, inter=768),
        dict(name="decode_moe", kind="moe", s=8, hidden=2048, experts=128, top_k=8, inter=768),
        # a caller that keeps its tensors in host memory: a Q8_0 projection of a few paragraphs
        dict(name="host_linear_q8", kind="host_linear", m=700, k=1024, n=3072, weight="q8_0"),
    ]


def _log_int(rng, lo, hi):
    """Whole numbers of [lo, hi], even over their logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


FLOPS = 9.9e10  # the most that the listed cases ask for


def draw(rng):
    kind = rng.choice(["mlp_w8a8", "mlp_f16", "attn_layer", "linear_i8", "linear_f16", "vision", "attention", "moe",
                       "host_linear"])
    if kind in ("mlp_w8a8", "mlp_f16"):
        hidden, inter = rng.choice([(1024, 3072), (768, 1152), (1152, 4304 if kind == "mlp_f16" else 4320), (2048, 768)])
        return dict(kind=kind, m=_log_int(rng, 1, min(3633, int(FLOPS / (6 * hidden * inter)))), hidden=hidden,
                    inter=inter, glu=rng.choice(["silu", "gelu"]))
    if kind == "attn_layer":
        h, kv, d = rng.choice([(16, 8, 128), (32, 4, 128), (16, 4, 64), (3, 1, 256)])
        return dict(kind=kind, s=_log_int(rng, 1, 3633 if h < 32 else 1500), hidden=rng.choice([768, 1024]), h=h, kv=kv, d=d)
    if kind in ("linear_i8", "linear_f16"):
        k, n = rng.choice([(1024, 3072), (3072, 1024), (1152, 3456), (1152, 1152), (1024, 1000), (2048, 4096)])
        c = dict(kind=kind, m=_log_int(rng, 1, 3633), k=k, n=n)
        if kind == "linear_i8":
            c["group"] = rng.choice([32, 64, 128])
        return c
    if kind == "vision":
        return dict(kind=kind, s=_log_int(rng, 60, 2394), hidden=1152, h=16, d=72, mlp=4304)
    if kind == "attention":
        h, kv, d = rng.choice([(16, 8, 128), (32, 4, 128), (16, 16, 72), (16, 4, 64), (3, 1, 256), (8, 8, 96)])
        if rng.random() < 0.5:  # a whole sequence
            n_q = n_kv = _log_int(rng, 5, min(4096, int(math.sqrt(FLOPS / (4 * h * d)))))
        else:  # its last queries against all its keys: a chunk of a long document, or one generated token
            n_kv = _log_int(rng, 30, 4096)
            n_q = _log_int(rng, 1, min(n_kv, 1024))
        mode = rng.choice(["causal", "causal", "none", "window", "causal_window"])
        return dict(kind=kind, n_q=n_q, n_kv=n_kv, h=h, kv=kv, d=d, mode=mode,
                    window=rng.choice([128, 512]) if "window" in mode else -1)
    if kind == "moe":
        hidden, experts, inter = rng.choice([(2048, 128, 768), (1024, 64, 512), (1024, 32, 768)])
        return dict(kind=kind, s=_log_int(rng, 1, 1024), hidden=hidden, experts=experts, top_k=rng.choice([4, 8]),
                    inter=inter)
    k, n = rng.choice([(1024, 3072), (3072, 1024), (1152, 1152)])
    return dict(kind=kind, m=_log_int(rng, 1, 700), k=k, n=n, weight=rng.choice(["f16", "q8_0", "i8", "qat", "qat_dynamic"]))


# ------------------------------------------------------------------ inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _weight(g, n, k):
    """An [n, k] weight as checkpoints hold it, N(0, 0.02²)."""
    return _randn(g, n, k, std=0.02)


def _host(t):
    return t.cpu().numpy()


def _norm_w(g, d):
    return (1.0 + 0.1 * torch.randn(d, generator=g, device="cuda")).half()


def _rope(s, d):
    ang = torch.arange(s, device="cuda", dtype=torch.float64)[:, None] * (
        10000.0 ** (-torch.arange(d // 2, device="cuda", dtype=torch.float64) / (d // 2)))[None, :]
    return ang.cos().half().contiguous(), ang.sin().half().contiguous()


def _q8_0(w):
    """Q8_0 of w [.., k]: (int8 codes [.., k/32, 32], fp16 scale [.., k/32])."""
    b = w.reshape(*w.shape[:-1], w.shape[-1] // 32, 32)
    d = (b.abs().amax(-1) / 127.0).half()
    inv = torch.where(d > 0, 1.0 / d.float(), torch.zeros_like(d, dtype=torch.float32))
    v = b * inv[..., None]
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)).clamp(-127, 127).to(torch.int8), d


def _q8_0_blocks(w):
    """w as GGUF holds it: 34-byte blocks."""
    q, d = _q8_0(w)
    return torch.cat([d.contiguous().view(torch.uint8).reshape(*d.shape, 2), q.view(torch.uint8)], -1).contiguous()


def _dequant(w):
    q, d = _q8_0(w)
    return (q.double() * d.double()[..., None]).reshape(w.shape)


def _quant64(x, group):
    """The activation quantizer in 64 bits: (codes, scales) per row and group."""
    b = x.reshape(x.shape[0], x.shape[1] // group, group)
    s = (b.abs().amax(-1) / 127.0).clamp_min(1e-12)
    v = b / s[..., None]
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)).clamp(-127, 127), s


def _deq64(x, group):
    q, s = _quant64(x, group)
    return (q * s[..., None]).reshape(x.shape)


def _inputs(c, seed):
    """The case's tensors, the same for prepare() and exact()."""
    g = _gen(seed)
    kind = c["kind"]
    t = {}
    if kind in ("mlp_w8a8", "mlp_f16"):
        t["x"] = _randn(g, c["m"], c["hidden"], dtype=torch.float16)
        t["nw"] = _norm_w(g, c["hidden"])
        t["gate"], t["up"] = _weight(g, c["inter"], c["hidden"]), _weight(g, c["inter"], c["hidden"])
        t["down"] = _weight(g, c["hidden"], c["inter"])
    elif kind == "attn_layer":
        t["x"] = _randn(g, c["s"], c["hidden"], dtype=torch.float16)
        t["nw"] = _norm_w(g, c["hidden"])
        t["qkv"] = _weight(g, (c["h"] + 2 * c["kv"]) * c["d"], c["hidden"])
        t["out"] = _weight(g, c["hidden"], c["h"] * c["d"])
        t["qw"], t["kw"] = _norm_w(g, c["d"]), _norm_w(g, c["d"])
        t["cos"], t["sin"] = _rope(c["s"], c["d"])
    elif kind in ("linear_i8", "linear_f16"):
        t["x"] = _randn(g, c["m"], c["k"], dtype=torch.float32 if kind == "linear_i8" else torch.float16)
        t["w"] = _weight(g, c["n"], c["k"])
    elif kind == "vision":
        t["x"] = _randn(g, c["s"], c["hidden"], dtype=torch.float16)
        for name, n, k in (("qkv", 3 * c["hidden"], c["hidden"]), ("out", c["hidden"], c["hidden"]),
                           ("fc1", c["mlp"], c["hidden"]), ("fc2", c["hidden"], c["mlp"])):
            t[name] = _weight(g, n, k)
    elif kind == "attention":
        t["q"] = _randn(g, c["n_q"], c["h"] * c["d"], dtype=torch.float16)
        t["k"] = _randn(g, c["n_kv"], c["kv"] * c["d"], dtype=torch.float16)
        t["v"] = _randn(g, c["n_kv"], c["kv"] * c["d"], dtype=torch.float16)
    elif kind == "moe":
        e, h, i = c["experts"], c["hidden"], c["inter"]
        t["x"] = _randn(g, c["s"], h)
        t["logits"] = _randn(g, c["s"], e)
        t["gate"], t["up"], t["down"] = (_randn(g, e, i, h, std=0.02), _randn(g, e, i, h, std=0.02),
                                         _randn(g, e, h, i, std=0.02))
    else:
        t["x"] = _randn(g, c["m"], c["k"])
        t["w"] = _weight(g, c["n"], c["k"])
        if c["weight"].startswith("qat"):
            t["codes"] = torch.randint(-127, 128, (c["n"], c["k"]), generator=g, device="cuda", dtype=torch.int8)
            t["ws"] = 3e-4 * (0.5 + torch.rand(c["n"], generator=g, device="cuda"))
    return t


# The static activation grid of a QAT layer whose inputs are N(0, 1): ±4 over the int8 range.
QAT_IN_SCALE = 4.0 / 127.0
MODES = {"none": rk.MASK_NONE, "causal": rk.MASK_CAUSAL, "window": rk.MASK_WINDOW, "causal_window": rk.MASK_CAUSAL_WINDOW}
GLU = {"silu": rk.GLU_SILU, "gelu": rk.GLU_GELU}


def _buf(*shape, dtype):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    rk.init(0)
    lib = rk.lib()
    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    s = dict(c=c, lib=lib, t=t)
    f16, f32, i8 = torch.float16, torch.float32, torch.int8
    if kind == "mlp_w8a8":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        s["glu"] = rk.pack_q8_0_glu(_host(_q8_0_blocks(t["gate"])), _host(_q8_0_blocks(t["up"])), inter, hid)
        s["down"] = rk.pack_q8_0(_host(_q8_0_blocks(t["down"])), hid, inter)
        s.update(q=_buf(m, hid, dtype=i8), qs=_buf(m, dtype=f32), act=_buf(m, inter, dtype=f32),
                 q2=_buf(m, inter, dtype=i8), qs2=_buf(m, dtype=f32), y=_buf(m, hid, dtype=f32))
    elif kind == "mlp_f16":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        s["glu"] = rk.pack_f16_glu(_host(t["gate"]), _host(t["up"]))
        s["down"] = rk.pack(_host(t["down"]))
        s.update(n=_buf(m, hid, dtype=f16), act=_buf(m, inter, dtype=f16), y=_buf(m, hid, dtype=f16))
    elif kind == "attn_layer":
        n, hd = c["s"], c["h"] * c["d"]
        s["wqkv"], s["wout"] = rk.pack(_host(t["qkv"])), rk.pack(_host(t["out"]))
        s.update(n=_buf(n, c["hidden"], dtype=f16), qkv=_buf(n, (c["h"] + 2 * c["kv"]) * c["d"], dtype=f16),
                 o=_buf(n, hd, dtype=f16), y=_buf(n, c["hidden"], dtype=f16))
    elif kind == "linear_i8":
        s["w"] = rk.pack_i8(_host(t["w"]), c["group"])
        s.update(q=_buf(c["m"], c["k"], dtype=i8), qs=_buf(c["m"], c["k"] // c["group"], dtype=f32),
                 y=_buf(c["m"], c["n"], dtype=f32))
    elif kind == "linear_f16":
        s["w"] = rk.pack(_host(t["w"]))
        s["y"] = _buf(c["m"], c["n"], dtype=f16)
    elif kind == "vision":
        n, hid = c["s"], c["hidden"]
        for name in ("qkv", "out", "fc1", "fc2"):
            s[name] = rk.pack(_host(t[name]))
        s.update(b=_buf(n, 3 * hid, dtype=f16), o=_buf(n, hid, dtype=f16), a=_buf(n, hid, dtype=f16),
                 m=_buf(n, c["mlp"], dtype=f16), y=_buf(n, hid, dtype=f16))
    elif kind == "attention":
        s["o"] = _buf(c["n_q"], c["h"] * c["d"], dtype=f16)
    elif kind == "moe":
        blocks = [_host(_q8_0_blocks(t.pop(k))) for k in ("gate", "up", "down")]
        s["w"] = rk.pack_moe_q8_0(*blocks, c["experts"], c["hidden"], c["inter"])
        ids, wts = rk.moe_route(_host(t["logits"]), c["top_k"])
        s.update(ids=np.ascontiguousarray(ids), wts=np.ascontiguousarray(wts), y=_buf(c["s"], c["hidden"], dtype=f32))
    else:
        w = c["weight"]
        if w == "f16":
            s["w"] = rk.pack(_host(t["w"]))
        elif w == "q8_0":
            s["w"] = rk.pack_q8_0(_host(_q8_0_blocks(t["w"])), c["n"], c["k"])
        elif w == "i8":
            s["w"] = rk.pack_i8(_host(t["w"]), 128)
        else:
            s["w"] = rk.pack_qat(_host(t["codes"]), _host(t["ws"]), c["n"], c["k"],
                                 QAT_IN_SCALE if w == "qat" else 0.0, 0.0)
        s["x"] = _host(t["x"])
        t.clear()
    # weights are resident now; the f32 sources are not part of the state
    for k in ("gate", "up", "down", "w", "codes"):
        t.pop(k, None)
    if kind in ("attn_layer", "vision"):
        for k in ("qkv", "out", "fc1", "fc2"):
            t.pop(k, None)
    torch.cuda.synchronize()  # the inputs come from torch's stream, the calls run on the library's
    return s


def _ok(rc):
    if rc != 0:
        raise RuntimeError(rk.lib().rk_last_error().decode())


def run(state):
    s, c, lib, t = state, state["c"], state["lib"], state["t"]
    kind = c["kind"]
    p = lambda x: x.data_ptr()  # noqa: E731
    F16, F32 = rk.DTYPE_F16, rk.DTYPE_F32
    if kind == "mlp_w8a8":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        _ok(lib.rk_rms_norm_quantize_dev(p(t["x"]), p(t["nw"]), F16, m, hid, EPS, F16, p(s["q"]), p(s["qs"]), None))
        _ok(lib.rk_matmul_w8a8_glu_dev(s["glu"], p(s["q"]), p(s["qs"]), m, hid, GLU[c["glu"]], p(s["act"]), 0, None))
        _ok(lib.rk_quantize_rows_dev(p(s["act"]), m, inter, inter, p(s["q2"]), p(s["qs2"]), None))
        _ok(lib.rk_matmul_w8a8_dev(s["down"], p(s["q2"]), p(s["qs2"]), inter, m, inter, p(s["y"]), None))
        return {"act": s["act"], "y": s["y"]}
    if kind == "mlp_f16":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        _ok(lib.rk_rms_norm_dev(p(t["x"]), p(t["nw"]), F16, p(s["n"]), m, hid, EPS, F16, None))
        _ok(lib.rk_matmul_f16_glu_dev(s["glu"], p(s["n"]), m, hid, GLU[c["glu"]], p(s["act"]), 1, None))
        _ok(lib.rk_matmul_f16_dev(s["down"], p(s["act"]), m, inter, p(s["y"]), None))
        return {"act": s["act"], "y": s["y"]}
    if kind == "attn_layer":
        n, h, kv, d = c["s"], c["h"], c["kv"], c["d"]
        _ok(lib.rk_rms_norm_dev(p(t["x"]), p(t["nw"]), F16, p(s["n"]), n, c["hidden"], EPS, F16, None))
        _ok(lib.rk_matmul_f16_dev(s["wqkv"], p(s["n"]), n, c["hidden"], p(s["qkv"]), None))
        _ok(lib.rk_attention_qkv_dev(p(s["qkv"]), n, (h + 2 * kv) * d, h, kv, d, p(t["qw"]), p(t["kw"]), EPS,
                                     p(t["cos"]), p(t["sin"]), F16, d ** -0.5, 0.0, rk.MASK_CAUSAL, -1, 0, 0,
                                     p(s["o"]), h * d, None))
        _ok(lib.rk_matmul_f16_dev(s["wout"], p(s["o"]), n, h * d, p(s["y"]), None))
        return {"o": s["o"], "y": s["y"]}
    if kind == "linear_i8":
        m, k, g = c["m"], c["k"], c["group"]
        _ok(lib.rk_quantize_rows_dev(p(t["x"]), m, k, g, p(s["q"]), p(s["qs"]), None))
        _ok(lib.rk_matmul_w8a8_dev(s["w"], p(s["q"]), p(s["qs"]), g, m, k, p(s["y"]), None))
        return s["y"]
    if kind == "linear_f16":
        _ok(lib.rk_matmul_f16_dev(s["w"], p(t["x"]), c["m"], c["k"], p(s["y"]), None))
        return s["y"]
    if kind == "vision":
        n, hid, h, d = c["s"], c["hidden"], c["h"], c["d"]
        _ok(lib.rk_matmul_f16_dev(s["qkv"], p(t["x"]), n, hid, p(s["b"]), None))
        b = p(s["b"])
        _ok(lib.rk_attention_strided_dev(b, 3 * hid, b + 2 * hid, 3 * hid, b + 4 * hid, 3 * hid, n, n, h, h, d,
                                         d ** -0.5, 0.0, rk.MASK_NONE, -1, 0, 0, p(s["o"]), hid, None))
        _ok(lib.rk_matmul_f16_dev(s["out"], p(s["o"]), n, hid, p(s["a"]), None))
        # fc1 and fc2 back to back: the activation between them belongs to the caller
        _ok(lib.rk_matmul_f16_dev(s["fc1"], p(s["a"]), n, hid, p(s["m"]), None))
        _ok(lib.rk_matmul_f16_dev(s["fc2"], p(s["m"]), n, c["mlp"], p(s["y"]), None))
        return {"o": s["o"], "a": s["a"], "m": s["m"], "y": s["y"]}
    if kind == "attention":
        _ok(lib.rk_attention_dev(p(t["q"]), p(t["k"]), p(t["v"]), c["n_q"], c["n_kv"], c["h"], c["kv"], c["d"],
                                 c["d"] ** -0.5, 0.0, MODES[c["mode"]], c["window"], c["n_kv"] - c["n_q"], 0,
                                 p(s["o"]), None))
        return s["o"]
    if kind == "moe":
        _ok(lib.rk_moe_experts_dev(s["w"], p(t["x"]), c["s"], c["top_k"], s["ids"].ctypes.data_as(ctypes.c_void_p),
                                   s["wts"].ctypes.data_as(ctypes.c_void_p), p(s["y"]), None))
        return s["y"]
    return rk.matmul(s["x"], s["w"])


# -------------------------------------------------------- what it comes to ----
def _pairs(c):
    """Visible (query, key) pairs."""
    t = np.arange(c["n_q"], dtype=np.int64) + c["n_kv"] - c["n_q"]
    lo, hi = np.zeros_like(t), np.full_like(t, c["n_kv"] - 1)
    w = c["window"]
    if c["mode"] == "causal":
        hi = t
    elif c["mode"] == "window":
        lo, hi = np.maximum(0, t - w), np.minimum(c["n_kv"] - 1, t + w)
    elif c["mode"] == "causal_window":
        lo, hi = np.maximum(0, t - w + 1), t
    return int((hi - lo + 1).sum())


Q8 = 34 / 32  # bytes of a Q8_0 value


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp_w8a8":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        return dict(bytes=2 * m * hid + 3 * hid * inter * Q8 + 4 * m * inter + 4 * m * hid, flops=6 * m * hid * inter)
    if kind == "mlp_f16":
        m, hid, inter = c["m"], c["hidden"], c["inter"]
        return dict(bytes=2 * m * hid + 6 * hid * inter + 2 * m * inter + 2 * m * hid, flops=6 * m * hid * inter)
    if kind == "attn_layer":
        n, hid, h, kv, d = c["s"], c["hidden"], c["h"], c["kv"], c["d"]
        wq, hd = (h + 2 * kv) * d, h * d
        return dict(bytes=4 * n * hid + 2 * hid * (wq + hd) + 2 * n * hd,
                    flops=2 * n * hid * (wq + hd) + 2 * d * h * n * (n + 1))
    if kind in ("linear_i8", "linear_f16"):
        m, k, n = c["m"], c["k"], c["n"]
        if kind == "linear_f16":
            return dict(bytes=2 * (m * k + n * k + m * n), flops=2 * m * n * k)
        return dict(bytes=4 * m * k + n * k * (1 + 4 / c["group"]) + 4 * m * n, flops=2 * m * n * k)
    if kind == "vision":
        n, hid, mlp, h, d = c["s"], c["hidden"], c["mlp"], c["h"], c["d"]
        return dict(bytes=2 * (n * hid + hid * (4 * hid + 2 * mlp) + n * (3 * hid + mlp)),
                    flops=2 * n * hid * (4 * hid + 2 * mlp) + 4 * n * n * h * d)
    if kind == "attention":
        return dict(bytes=2 * c["d"] * (2 * c["n_q"] * c["h"] + 2 * c["n_kv"] * c["kv"]),
                    flops=4 * c["d"] * c["h"] * _pairs(c))
    if kind == "moe":
        s, hid, inter, k, e = c["s"], c["hidden"], c["inter"], c["top_k"], c["experts"]
        used = e * (1 - (1 - k / e) ** s)  # experts that some token is routed to, on average
        return dict(bytes=used * 3 * hid * inter * Q8 + 8 * s * hid, flops=6 * s * k * hid * inter)
    m, k, n = c["m"], c["k"], c["n"]
    return dict(bytes=4 * m * k + n * k * {"f16": 2, "q8_0": Q8}.get(c["weight"], 1) + 4 * m * n, flops=2 * m * n * k)


def tolerance(case):
    kind = case["kind"]
    # four times what another order of the sums shows, per kind (fp16 results: one rounding of 2^-11; re-quantized
    # activations: a code that a last-bit difference moves by one is 1/127 of its row's largest value)
    if kind in ("mlp_w8a8", "moe"):
        return {"rel": 2e-3, "max": 0.2}
    if kind == "linear_i8":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "host_linear":
        return {"rel": 1e-3, "max": 0.02} if case["weight"] == "f16" else {"rel": 1e-5, "max": 1e-3}
    return {"rel": 2e-3, "max": 0.05}


# ------------------------------------------------------------- in 64 bits ----
def _rms64(x, w):
    x = x.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _glu64(g, u, glu):
    if glu == "silu":
        return g * torch.sigmoid(g) * u
    return 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u


def _half64(w):
    return w.half().double()


def _attention64(q, k, v, h, kv, d, mode, window, q0):
    """q [n_q, h·d], k / v [n_kv, kv·d] in 64 bits, query rows in chunks."""
    n_q, n_kv = q.shape[0], k.shape[0]
    k = k.reshape(n_kv, kv, d).permute(1, 2, 0).contiguous()
    v = v.reshape(n_kv, kv, d).permute(1, 0, 2).contiguous()
    out = torch.empty(n_q, h, d, dtype=torch.float64, device=q.device)
    j = torch.arange(n_kv, device=q.device)[None, :]
    for a in range(0, n_q, 512):
        b = min(n_q, a + 512)
        t = torch.arange(a, b, device=q.device)[:, None] + q0
        see = torch.ones(b - a, n_kv, dtype=torch.bool, device=q.device)
        if "causal" in mode:
            see &= j <= t
        if mode == "window":
            see &= (t - j).abs() <= window
        if mode == "causal_window":
            see &= j > t - window
        for i in range(h):
            g = i // (h // kv)
            sc = (q[a:b].reshape(b - a, h, d)[:, i] @ k[g]) * d ** -0.5
            out[a:b, i] = torch.softmax(sc.masked_fill(~see, -math.inf), -1) @ v[g]
    return out.reshape(n_q, h * d)


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "mlp_w8a8":
        # the norm's fp16 result and the int8 codes are what the path defines; all sums in 64 bits
        n = _deq64(_rms64(t["x"], t["nw"]).half().double(), c["hidden"])
        act = _glu64(n @ _dequant(t["gate"]).T, n @ _dequant(t["up"]).T, c["glu"])
        return {"act": act, "y": _deq64(act, c["inter"]) @ _dequant(t["down"]).T}
    if kind == "mlp_f16":
        n = _rms64(t["x"], t["nw"])
        act = _glu64(n @ _half64(t["gate"]).T, n @ _half64(t["up"]).T, c["glu"])
        return {"act": act, "y": act @ _half64(t["down"]).T}
    if kind == "attn_layer":
        n, h, kv, d = c["s"], c["h"], c["kv"], c["d"]
        qkv = _rms64(t["x"], t["nw"]) @ _half64(t["qkv"]).T
        q, k, v = qkv.split([h * d, kv * d, kv * d], 1)

        def head(x, w):
            x = _rms64(x.reshape(n, -1, d), w)
            cs, sn = t["cos"].double()[:, None], t["sin"].double()[:, None]
            a, b = x[..., :d // 2], x[..., d // 2:]
            return torch.cat([a * cs - b * sn, b * cs + a * sn], -1).reshape(n, -1)
        o = _attention64(head(q, t["qw"]), head(k, t["kw"]), v, h, kv, d, "causal", -1, 0)
        return {"o": o, "y": o @ _half64(t["out"]).T}
    if kind == "linear_i8":
        return _deq64(t["x"].double(), c["group"]) @ _deq64(t["w"].double(), c["group"]).T
    if kind == "linear_f16":
        return t["x"].double() @ _half64(t["w"]).T
    if kind == "vision":
        hid, h, d = c["hidden"], c["h"], c["d"]
        q, k, v = (t["x"].double() @ _half64(t["qkv"]).T).split(hid, 1)
        o = _attention64(q, k, v, h, h, d, "none", -1, 0)
        a = o @ _half64(t["out"]).T
        m = a @ _half64(t["fc1"]).T
        return {"o": o, "a": a, "m": m, "y": m @ _half64(t["fc2"]).T}
    if kind == "attention":
        return _attention64(t["q"].double(), t["k"].double(), t["v"].double(), c["h"], c["kv"], c["d"], c["mode"],
                            c["window"], c["n_kv"] - c["n_q"])
    if kind == "moe":
        x = _deq64(t["x"].double(), 32)
        top, ids = torch.softmax(t["logits"].double(), -1).topk(c["top_k"], -1)
        wts = top / top.sum(-1, keepdim=True)
        y = torch.zeros(c["s"], c["hidden"], dtype=torch.float64, device=x.device)
        for e in range(c["experts"]):
            rows, slot = (ids == e).nonzero(as_tuple=True)
            if not rows.numel():
                continue
            act = _glu64(x[rows] @ _dequant(t["gate"][e]).T, x[rows] @ _dequant(t["up"][e]).T, "silu")
            y[rows] += wts[rows, slot][:, None] * (_deq64(act, 32) @ _dequant(t["down"][e]).T)
        return y
    x, w = t["x"].double(), c["weight"]
    if w == "f16":
        return _host(x.half().double() @ _half64(t["w"]).T)
    if w == "q8_0":
        return _host(_deq64(x, 32) @ _dequant(t["w"]).T)
    if w == "i8":
        return _host(_deq64(x, 128) @ _deq64(t["w"].double(), 128).T)
    s = QAT_IN_SCALE if w == "qat" else (x.abs().amax(-1, keepdim=True) / 127.0).clamp_min(1e-12)
    q = torch.round(x / s).clamp(-128, 127)
    return _host((q @ t["codes"].double().T) * (s * t["ws"].double()[None, :]))
