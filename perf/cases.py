"""Workloads of the quantized decode path as an engine has it do them, through the public entry points.

Six kinds of work, at Llama-3-8B shapes (hidden 4096, 32 q / 8 kv heads, head 128, MLP 14336) and at the per-GPU shapes of
Llama-3-70B on eight GPUs (hidden 8192, 8 q / 1 kv heads, MLP 3584):

  decode   ``PagedAttention.forward_decode``: one new token per sequence over a paged cache in the x layout
  engine   ``TritonAttentionImpl.forward``: cache write + attention of one engine step (decode tokens, prefill chunks or both)
  prefix   ``PagedAttention.write_to_paged_cache`` + ``forward_prefix``: chunked prefill over a cached prefix, x layout
  linear   ``PTPCFp8LinearMethod.apply``: per-token quantisation + fp8 GEMM
  mlp      residual add + RMSNorm + quantisation, gate/up GEMM, SiLU-mul + quantisation, down GEMM
  step     one decoder layer of a decode step (without the rotary embedding), replayed from a captured graph
"""
from __future__ import annotations

import math
import types

import torch

from vllm_amd import _custom_ops as ops
from vllm_amd.attention import PagedAttention
from vllm_amd.quantization import PTPCFp8LinearMethod
from vllm_amd.v1.attention.backends.triton_attn import TritonAttentionBackend, TritonAttentionImpl, TritonAttentionMetadata

DEV = "cuda"
FP8 = torch.float8_e4m3fn
EPS = 1e-5
KV_SCALE = 0.25      # calibrated per-tensor scale of an fp8 cache
SILU_SCALE = 0.02    # static activation scale in front of the down projection
NORM_SCALE = 0.02    # static activation scale in front of the gate/up projection
CAPTURE_LEN = 8192   # max_seq_len an engine captures its decode graphs with


def listed():
    return [
        # one user's chat turn: a single sequence, a few hundred tokens -- latency and launches
        {"name": "decode_one", "kind": "decode", "seqs": 1, "ctx": 777, "ragged": False, "heads": 32, "kv_heads": 8,
         "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
        # the headline: a full decode batch at one context length
        {"name": "decode_batch", "kind": "decode", "seqs": 64, "ctx": 4096, "ragged": False, "heads": 32, "kv_heads": 8,
         "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
        # continuous batching: every sequence at its own length, unquantised cache
        {"name": "decode_ragged", "kind": "decode", "seqs": 45, "ctx": 4001, "ragged": True, "heads": 32, "kv_heads": 8,
         "head": 128, "block": 16, "kv": "auto", "dtype": "bf16"},
        # long documents: few sequences, the keys split over the chip
        {"name": "decode_long", "kind": "decode", "seqs": 8, "ctx": 131072, "ragged": False, "heads": 64, "kv_heads": 8,
         "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
        # a decode step of the V1 engine's backend, write of the new token included
        {"name": "engine_decode", "kind": "engine", "chunks": 0, "new": 0, "cached": 0, "decodes": 61, "ctx": 3000,
         "ragged": True, "heads": 32, "kv_heads": 8, "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
        # a step of that engine with one prefill chunk among running decodes
        {"name": "engine_mixed", "kind": "engine", "chunks": 1, "new": 2000, "cached": 1500, "decodes": 63, "ctx": 4096,
         "ragged": True, "heads": 32, "kv_heads": 8, "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
        # two long prompts from scratch, unquantised cache
        {"name": "engine_prefill", "kind": "engine", "chunks": 2, "new": 5003, "cached": 0, "decodes": 0, "ctx": 0,
         "ragged": True, "heads": 32, "kv_heads": 8, "head": 128, "block": 16, "kv": "auto", "dtype": "bf16"},
        # many short chunks over long cached prefixes (shared system prompts)
        {"name": "prefix_chunks", "kind": "prefix", "chunks": 24, "new": 250, "cached": 3000, "ragged": True, "heads": 32,
         "kv_heads": 8, "head": 128, "block": 16, "kv": "fp8", "dtype": "fp16"},
        # one projection of a small decode batch
        {"name": "linear_small", "kind": "linear", "tokens": 17, "k": 4096, "n": 6144, "dtype": "bf16"},
        # the MLP of one chunked-prefill step of a tensor-parallel rank
        {"name": "mlp_chunk", "kind": "mlp", "tokens": 509, "hidden": 8192, "inter": 3584, "act": "token", "dtype": "bf16"},
        # the MLP of a long prefill
        {"name": "mlp_prefill", "kind": "mlp", "tokens": 4096, "hidden": 4096, "inter": 14336, "act": "token", "dtype": "bf16"},
        # one layer of a decode step, replayed from the engine's captured graph
        {"name": "step_graph", "kind": "step", "seqs": 32, "ctx": 1500, "hidden": 4096, "inter": 14336, "heads": 32,
         "kv_heads": 8, "head": 128, "block": 16, "kv": "fp8", "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "engine", "engine", "prefix", "linear", "mlp", "step"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "linear":
        k, n = rng.choice([(4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096), (1024, 8192), (3584, 8192), (8192, 1280),
                           (8192, 7168)])
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "k": k, "n": n, "dtype": dtype}
    if kind == "mlp":
        hidden, inter = rng.choice([(4096, 14336), (8192, 3584)])
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "hidden": hidden, "inter": inter,
                "act": rng.choice(["token", "token", "static"]), "dtype": dtype}
    if kind == "step":
        hidden, inter, heads, kv_heads = rng.choice([(4096, 14336, 32, 8), (8192, 3584, 8, 1)])
        return {"kind": kind, "seqs": _log(rng, 1, 128), "ctx": _log(rng, 100, 4096), "hidden": hidden, "inter": inter,
                "heads": heads, "kv_heads": kv_heads, "head": 128, "block": 16, "kv": rng.choice(["fp8", "auto"]), "dtype": "bf16"}
    heads, kv_heads, head = rng.choice([(32, 8, 128), (32, 8, 128), (8, 1, 128), (64, 8, 128), (32, 8, 64), (16, 8, 256)])
    kv = rng.choice(["fp8", "fp8", "auto"])
    # keys of the whole batch within 1 GiB of cache, half of the largest listed one
    most = (1 << 30) // (2 * kv_heads * head * (1 if kv == "fp8" else 2))
    case = {"kind": kind, "ragged": rng.random() < 0.7, "heads": heads, "kv_heads": kv_heads, "head": head,
            "block": rng.choice([16, 16, 32]), "kv": kv, "dtype": dtype}
    if kind == "decode":
        seqs = _log(rng, 1, 256)
        return {**case, "seqs": seqs, "ctx": _log(rng, 64, min(131072, most // seqs))}
    # query x key pairs of the chunks: within those of two prompts of 5000 tokens per 32 heads of 128
    chunks, new, cached = _log(rng, 1, 32), _log(rng, 33, 6000), rng.choice([0, _log(rng, 64, 8192)])
    while chunks * new * (cached + new / 2) * heads * head > 1.2e11:
        chunks, new, cached = max(1, chunks // 2), (new + 1) // 2 if chunks == 1 else new, cached * 3 // 4
    if kind == "prefix":
        return {**case, "chunks": chunks, "new": new, "cached": cached}
    form = rng.choice(["decode", "mixed", "prefill"])
    if form == "decode":
        chunks = new = cached = 0
    decodes = 0 if form == "prefill" else _log(rng, 1, 200)
    ctx = 0 if not decodes else _log(rng, 64, min(16384, most // (2 * decodes)))
    return {**case, "chunks": chunks, "new": new, "cached": cached, "decodes": decodes, "ctx": ctx}


# ---- lengths: a function of the case alone, so that the work is too ------------------------------------------------------
def _spread(n, top, low, ragged):
    """n lengths up to `top`: all alike, or spread evenly over [low * top, top] in an order that is not sorted."""
    if not ragged or n == 1:
        return [top] * n
    ls = [max(1, int(top * (low + (1 - low) * i / (n - 1)))) for i in range(n)]
    step = next(s for s in range(max(1, n // 3), n + 2) if math.gcd(s, n) == 1)
    return [ls[(i * step) % n] for i in range(n)]


def _batch(c):
    """(query length, total length) of every sequence of the step, decode tokens first as an engine orders them."""
    if c["kind"] in ("decode", "step"):
        return [(1, n) for n in _spread(c["seqs"], c["ctx"], 0.125, c.get("ragged", True))]
    rows = [(1, n) for n in _spread(c.get("decodes", 0), c.get("ctx", 0), 0.125, c["ragged"])]
    new = _spread(c["chunks"], c["new"], 0.6, c["ragged"])
    cached = _spread(c["chunks"], c["cached"], 0.5, c["ragged"])
    return rows + [(q, q + (p if c["cached"] else 0)) for q, p in zip(new, cached)]


def _dtype(c):
    return torch.bfloat16 if c["dtype"] == "bf16" else torch.float16


# ---- inputs ---------------------------------------------------------------------------------------------------------------
def _rand_cache(shape, c, g):
    """Keys / values of unit variance: fp8 codes under KV_SCALE (uint8), or the query's own type."""
    t = torch.empty(shape, dtype=torch.uint8 if c["kv"] == "fp8" else _dtype(c), device=DEV)
    for i in range(0, shape[0], 4096):
        part = torch.randn(t[i:i + 4096].shape, generator=g, device=DEV)
        if c["kv"] == "fp8":
            t[i:i + 4096] = (part / KV_SCALE).to(FP8).view(torch.uint8)
        else:
            t[i:i + 4096] = part
    return t


def _paged(c, g, layout):
    """Block table, cache and slots of the new tokens, blocks dealt at random as a running engine's are."""
    rows, bs, kvh, d = _batch(c), c["block"], c["kv_heads"], c["head"]
    need = [-(-n // bs) for _, n in rows]
    nb = sum(need)
    perm = torch.randperm(nb, generator=g, device=DEV).to(torch.int32)
    table = torch.zeros((len(rows), max(need)), dtype=torch.int32, device=DEV)
    at = 0
    for i, k in enumerate(need):
        table[i, :k] = perm[at:at + k]
        at += k
    if layout == "x":
        x = 16 if c["kv"] == "fp8" else 8
        k_cache = _rand_cache((nb, kvh, d // x, bs, x), c, g)
        v_cache = _rand_cache((nb, kvh, d, bs), c, g)
        cache = (k_cache, v_cache)
    else:
        order = TritonAttentionBackend.get_kv_cache_stride_order()
        shape = TritonAttentionBackend.get_kv_cache_shape(nb, bs, kvh, d)
        mem = torch.empty(tuple(shape[i] for i in order), dtype=torch.uint8 if c["kv"] == "fp8" else _dtype(c), device=DEV)
        for half in mem:
            half.copy_(_rand_cache(tuple(half.shape), c, g))
        cache = mem.permute(tuple(order.index(i) for i in range(5)))
    pos = torch.cat([torch.arange(n - q, n, device=DEV) for q, n in rows])
    seq = torch.repeat_interleave(torch.arange(len(rows), device=DEV), torch.tensor([q for q, _ in rows], device=DEV))
    slots = table[seq, pos // bs].to(torch.int64) * bs + pos % bs
    ql = torch.tensor([q for q, _ in rows], dtype=torch.int32)
    start = torch.zeros(len(rows) + 1, dtype=torch.int32)
    start[1:] = torch.cumsum(ql, 0)
    return dict(rows=rows, table=table, cache=cache, slots=slots, start=start.to(DEV),
                lens=torch.tensor([n for _, n in rows], dtype=torch.int32, device=DEV),
                max_q=max(q for q, _ in rows), max_len=max(n for _, n in rows))


def _randn(g, *shape, dtype, mul=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * mul).to(dtype)


def _inputs(c, seed):
    """Everything that is drawn at random, the same for run() and for exact()."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = _dtype(c)
    s = {}
    if c["kind"] in ("decode", "engine", "prefix", "step"):
        s.update(_paged(c, g, "flash" if c["kind"] == "engine" else "x"))
        s["scale"] = torch.tensor([KV_SCALE if c["kv"] == "fp8" else 1.0], dtype=torch.float32, device=DEV)
    if c["kind"] in ("decode", "engine", "prefix"):
        t = sum(q for q, _ in s["rows"])
        s["q"] = _randn(g, t, c["heads"], c["head"], dtype=dt)
        if c["kind"] != "decode":
            s["k"] = _randn(g, t, c["kv_heads"], c["head"], dtype=dt)
            s["v"] = _randn(g, t, c["kv_heads"], c["head"], dtype=dt)
    if c["kind"] == "linear":
        s["x"] = _randn(g, c["tokens"], c["k"], dtype=dt)
        s["w"] = _randn(g, c["n"], c["k"], dtype=torch.bfloat16, mul=c["k"] ** -0.5)
    if c["kind"] in ("mlp", "step"):
        h, i, t = c["hidden"], c["inter"], c["tokens"] if c["kind"] == "mlp" else c["seqs"]
        s["x"] = _randn(g, t, h, dtype=dt)
        s["res"] = _randn(g, t, h, dtype=dt, mul=3.0)
        s["norm"] = (1 + 0.1 * torch.randn(h, generator=g, device=DEV)).to(dt)
        s["w_up"] = _randn(g, 2 * i, h, dtype=torch.bfloat16, mul=h ** -0.5)
        s["w_down"] = _randn(g, h, i, dtype=torch.bfloat16, mul=i ** -0.5)
        if c["kind"] == "step":
            a = c["heads"] * c["head"]
            s["norm0"] = (1 + 0.1 * torch.randn(h, generator=g, device=DEV)).to(dt)
            s["w_qkv"] = _randn(g, a + 2 * c["kv_heads"] * c["head"], h, dtype=torch.bfloat16, mul=h ** -0.5)
            s["w_o"] = _randn(g, h, a, dtype=torch.bfloat16, mul=a ** -0.5)
    return s


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"] = c
    for name in ("w", "w_up", "w_down", "w_qkv", "w_o"):
        if name in s:
            s[name] = PTPCFp8LinearMethod.process_weights_after_loading(s[name])
    if c["kind"] == "linear":
        s["method"] = PTPCFp8LinearMethod()
    if c["kind"] in ("mlp", "step"):
        s["silu_scale"] = torch.tensor([SILU_SCALE], dtype=torch.float32, device=DEV)
        s["norm_scale"] = torch.tensor([NORM_SCALE], dtype=torch.float32, device=DEV)
    if c["kind"] == "engine":
        s["impl"] = TritonAttentionImpl(c["heads"], c["head"], c["head"] ** -0.5, c["kv_heads"], None, None, "fp8" if c["kv"] == "fp8" else "auto")
        s["layer"] = types.SimpleNamespace(_k_scale=s["scale"], _v_scale=s["scale"], _q_scale=1.0)
        s["meta"] = TritonAttentionMetadata(
            num_actual_tokens=s["q"].shape[0], max_query_len=s["max_q"], query_start_loc=s["start"], max_seq_len=s["max_len"],
            seq_lens=s["lens"], block_table=s["table"], slot_mapping=s["slots"], use_cascade=False, common_prefix_len=0,
            cu_prefix_query_lens=None, prefix_kv_lens=None, suffix_kv_lens=None)
        s["out"] = torch.empty_like(s["q"])
    if c["kind"] == "step":
        res = s["res"].clone()
        _layer(s)                       # the engine's warm-up pass in front of a capture
        s["graph"] = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(s["graph"]):
            s["hidden"] = _layer(s)
        s["res"].copy_(res)
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------------
def _mlp(s, x):
    c, dt = s["case"], x.dtype
    if c.get("act") == "static":
        qx, sx = torch.empty(x.shape, dtype=FP8, device=x.device), s["norm_scale"]
        ops.scaled_fused_add_rms_norm(qx, x, s["res"], s["norm"], sx, EPS)
    else:
        qx, sx = ops.rms_norm_dynamic_per_token_quant(x, s["norm"], EPS, FP8, None, s["res"])
    up = ops.cutlass_scaled_mm(qx, s["w_up"][0], sx, s["w_up"][1], dt)
    act = torch.empty((x.shape[0], c["inter"]), dtype=FP8, device=x.device)
    ops.silu_and_mul_quant(act, up, s["silu_scale"])
    return ops.cutlass_scaled_mm(act, s["w_down"][0], s["silu_scale"], s["w_down"][1], dt)


def _layer(s):
    c = s["case"]
    h, kvh, d, t = c["heads"], c["kv_heads"], c["head"], s["x"].shape[0]
    kv = "fp8" if c["kv"] == "fp8" else "auto"
    k_cache, v_cache = s["cache"]
    qx, sx = ops.rms_norm_dynamic_per_token_quant(s["x"], s["norm0"], EPS, FP8, None, s["res"])
    qkv = ops.cutlass_scaled_mm(qx, s["w_qkv"][0], sx, s["w_qkv"][1], s["x"].dtype)
    q, k, v = qkv.split([h * d, kvh * d, kvh * d], dim=1)
    PagedAttention.write_to_paged_cache(k.view(t, kvh, d), v.view(t, kvh, d), k_cache, v_cache, s["slots"], kv, s["scale"], s["scale"])
    a = PagedAttention.forward_decode(q.view(t, h, d), k_cache, v_cache, s["table"], s["lens"], CAPTURE_LEN, kv, kvh, d ** -0.5,
                                      None, s["scale"], s["scale"])
    qa, sa = ops.scaled_fp8_quant(a.view(t, h * d), use_per_token_if_dynamic=True)
    o = ops.cutlass_scaled_mm(qa, s["w_o"][0], sa, s["w_o"][1], s["x"].dtype)
    return _mlp(s, o)


def run(state):
    s, c = state, state["case"]
    kv = "fp8" if c.get("kv") == "fp8" else "auto"
    if c["kind"] == "decode":
        return PagedAttention.forward_decode(s["q"], *s["cache"], s["table"], s["lens"], s["max_len"], kv, c["kv_heads"],
                                             c["head"] ** -0.5, None, s["scale"], s["scale"])
    if c["kind"] == "engine":
        return {"out": s["impl"].forward(s["layer"], s["q"], s["k"], s["v"], s["cache"], s["meta"], s["out"]), "cache": s["cache"]}
    if c["kind"] == "prefix":
        PagedAttention.write_to_paged_cache(s["k"], s["v"], *s["cache"], s["slots"], kv, s["scale"], s["scale"])
        out = PagedAttention.forward_prefix(s["q"], s["k"], s["v"], kv, *s["cache"], s["table"], s["start"], s["lens"], s["max_q"],
                                            None, None, s["scale"], s["scale"])
        return {"out": out, "k_cache": s["cache"][0], "v_cache": s["cache"][1]}
    if c["kind"] == "linear":
        return s["method"].apply(*s["w"], s["x"])
    if c["kind"] == "mlp":
        return {"out": _mlp(s, s["x"]), "residual": s["res"]}
    s["graph"].replay()
    return {"out": s["hidden"], "residual": s["res"], "k_cache": s["cache"][0], "v_cache": s["cache"][1]}


# ---- the work of a pass, the tolerance, the result in 64 bits -----------------------------------------------------------
def work(case):
    c, el = case, 2
    if c["kind"] == "linear":
        m, k, n = c["tokens"], c["k"], c["n"]
        return {"bytes": m * k * el + k * n + 4 * n + m * n * el, "flops": 2 * m * n * k}
    total, flops = 0, 0
    if c["kind"] in ("mlp", "step"):
        m, h, i = c["tokens"] if c["kind"] == "mlp" else c["seqs"], c["hidden"], c["inter"]
        total += 3 * h * i + 4 * (2 * i + h) + 2 * h + m * h * el * 4      # weights, scales; x, residual in; out, residual out
        flops += 6 * m * h * i
        if c["kind"] == "mlp":
            return {"bytes": total, "flops": flops}
        a, b = c["heads"] * c["head"], c["kv_heads"] * c["head"]
        total += h * (a + 2 * b) + a * h + 4 * (a + 2 * b + h) + 2 * h
        flops += 2 * m * h * (2 * a + 2 * b)
    rows, b = _batch(c), 1 if c["kv"] == "fp8" else 2
    keys, queries = sum(n for _, n in rows), sum(q for q, _ in rows)
    total += 2 * keys * c["kv_heads"] * c["head"] * b + sum(-(-n // c["block"]) for _, n in rows) * 4
    if c["kind"] != "step":
        total += 2 * queries * c["heads"] * c["head"] * el
        if c["kind"] != "decode":
            total += 2 * queries * c["kv_heads"] * c["head"] * el + 8 * queries
    flops += 4 * c["heads"] * c["head"] * sum(q * (n - q) + q * (q + 1) // 2 for q, n in rows)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] in ("mlp", "step"):
        # chains with fp8 roundings between the products: a last bit upstream moves single codes (1.5e-2 .. 2.3e-2 against 64 bits)
        return {"rel": 3e-2, "max": 0.25, "differ": 2e-3}
    # the rounding of the result, and of the probabilities in front of the product with the values: 2.1e-3 .. 2.8e-3 against
    # 64 bits for bf16, 2.9e-4 for fp16
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 0.05}


def _q8(x, scale):
    """64-bit values -> the nearest e4m3 values of x / scale, in 64 bits."""
    return (x / scale).clamp(-448, 448).float().to(FP8).double()


def _w8(w):
    """A weight as the per-channel quantisation leaves it: (codes, scales) in 64 bits."""
    w = w.double()
    s = w.abs().amax(1, keepdim=True).float() / 448
    return _q8(w, s.double()), s.double()


def _mm(x, w, dt):
    """The product of per-token quantised rows and quantised weights, rounded to the type that the op returns."""
    codes, scales = w
    s = (x.abs().amax(1, keepdim=True) / 448).clamp_min(1 / (448 * 512))
    return ((_q8(x, s) @ codes.t()) * s * scales.t()).to(dt).double()


def _norm_mm(x, res, norm, w, dt, static):
    """Residual add, RMSNorm, quantisation, product: (product, residual)."""
    r = x + res
    stored = r.to(dt).double()
    if static:
        r = stored
    y = (r * torch.rsqrt(r.square().mean(1, keepdim=True) + EPS)).to(dt).double() * norm.double()
    if not static:
        return _mm(y.to(dt).double(), w, dt), stored
    return ((_q8(y, NORM_SCALE) @ w[0].t()) * NORM_SCALE * w[1].t()).to(dt).double(), stored


def _mlp64(s, c, x, res, dt):
    up, res = _norm_mm(x, res, s["norm"], _w8(s["w_up"]), dt, c.get("act") == "static")
    gate, lin = up[:, :c["inter"]], up[:, c["inter"]:]
    act = _q8(gate / (1 + torch.exp(-gate)) * lin, SILU_SCALE)
    codes, scales = _w8(s["w_down"])
    return (act @ codes.t()) * SILU_SCALE * scales.t(), res


def _attend64(s, c, q, new):
    """Causal attention of the step's rows over the paged cache. `new`: (k, v) of the step's own tokens as the queries see them."""
    h, kvh, d, bs = c["heads"], c["kv_heads"], c["head"], c["block"]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    scale = float(s["scale"][0])
    at = 0
    for i, (ql, n) in enumerate(s["rows"]):
        blocks = s["table"][i, :-(-n // bs)].long()
        if c["kind"] == "engine":
            k, v = (x[blocks].permute(2, 0, 1, 3).reshape(kvh, -1, d)[:, :n] for x in s["cache"])
        else:
            k = s["cache"][0][blocks].permute(1, 0, 3, 2, 4).reshape(kvh, -1, d)[:, :n]
            v = s["cache"][1][blocks].permute(1, 0, 3, 2).reshape(kvh, -1, d)[:, :n]
        if c["kv"] == "fp8":
            k, v = (x.contiguous().view(FP8).double() * scale for x in (k, v))
        else:
            k, v = k.double(), v.double()
        if new is not None:
            k, v = k.clone(), v.clone()
            k[:, n - ql:], v[:, n - ql:] = (x[at:at + ql].permute(1, 0, 2) for x in new)
        for r in range(0, ql, 2048):
            e = min(ql, r + 2048)
            hide = torch.arange(n, device=DEV)[None] > (n - ql + torch.arange(r, e, device=DEV))[:, None]
            for j in range(kvh):
                rows = q[at + r:at + e, j * (h // kvh):(j + 1) * (h // kvh)].double()
                sc = (rows.reshape(-1, d) @ k[j].t()).view(e - r, h // kvh, n) * d ** -0.5
                p = torch.softmax(sc.masked_fill_(hide[:, None], -math.inf), 2)
                out[at + r:at + e, j * (h // kvh):(j + 1) * (h // kvh)] = (p.view(-1, n) @ v[j]).view(e - r, h // kvh, d)
        at += ql
    return out


def _stored(x, c):
    """Keys / values as the cache holds them."""
    return _q8(x.double(), KV_SCALE) * KV_SCALE if c["kv"] == "fp8" else x.double()


def exact(case, seed):
    c, s, dt = case, _inputs(case, seed), _dtype(case)
    if c["kind"] == "linear":
        return _mm(s["x"].double(), _w8(s["w"]), torch.float64)
    if c["kind"] == "mlp":
        out, res = _mlp64(s, c, s["x"].double(), s["res"].double(), dt)
        return {"out": out, "residual": res}
    if c["kind"] == "decode":
        return _attend64(s, c, s["q"], None)
    if c["kind"] == "engine":
        return {"out": _attend64(s, c, s["q"], (_stored(s["k"], c), _stored(s["v"], c))), "cache": None}
    if c["kind"] == "prefix":     # the chunk's own keys are read as they came, before the cache rounds them
        return {"out": _attend64(s, c, s["q"], (s["k"].double(), s["v"].double())), "k_cache": None, "v_cache": None}
    h, kvh, d, t = c["heads"], c["kv_heads"], c["head"], c["seqs"]
    qkv, res = _norm_mm(s["x"].double(), s["res"].double(), s["norm0"], _w8(s["w_qkv"]), dt, False)
    q, k, v = qkv.split([h * d, kvh * d, kvh * d], dim=1)
    a = _attend64(s, c, q.view(t, h, d), (_stored(k.view(t, kvh, d), c), _stored(v.view(t, kvh, d), c)))
    o = _mm(a.reshape(t, h * d).to(dt).double(), _w8(s["w_o"]), dt)
    out, res = _mlp64(s, c, o, res, dt)
    return {"out": out, "residual": res, "k_cache": None, "v_cache": None}
