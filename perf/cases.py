"""The work a program gives this framework, as cases that can be timed: attention over prompts and over a KV cache, the
int8 layer for one token and for a prompt, and the end of the model that chooses the next token.

Every case goes through the public Python entry points (tscale_amd.AttentionContext, KVCache and the layer functions of
tscale_amd.attention).  Kinds of case:

  decode   one new query per sequence over a KV cache (generation, attention only)
  prefill  attention of whole prompts on 8-bit Q, K and V that a projection left in memory: one layer over the full
           causal window, or a pair of layers, a short window with ALiBi and the full one, as the layer schedule
           alternates them
  context  attention for a program with its own floating-point model: masks of a new batch, row quantisation of Q, K
           and V, attention, and the batch's rows into the KV cache
  token    one generated token per sequence: embedding, four int8 layers (two short-window / full-window pairs, the
           unit the layer schedule repeats) with the append to their caches, final normalisation; called one by one
           or recorded once as a HIP graph and replayed
  prompt   prompts through the embedding and one int8 layer in batch form, their rows into the layer's KV cache
  head     final layer's product, softmax over the vocabulary and the sampled choice
"""
import math
import random

import numpy as np
import torch

from tscale_amd import AttentionContext, KVCache, capi
from tscale_amd.attention import VEC_SCALE, add_lookup_product, add_lookup_product_prompt, flush_state

DTYPES = {"int8": capi.I8, "e4m3": capi.E4M3}
LAYERS = 4             # of a token step: two (short window, full window) pairs
SHORT_WINDOW = 64      # keys of a short-window layer of the model, slope SHORT_SLOPE
SHORT_SLOPE = 0.5
EMBED_ROWS = 50257     # labels of the embedding
# (heads, head width) of the attention that configurations use
SHAPES = ((12, 64), (16, 128), (8, 64), (16, 64), (8, 128), (12, 128))


def listed():
    return [
        # a chat with one user, early on: the latency of a single small call
        {"name": "decode-one", "kind": "decode", "dtype": "int8", "query": "8bit", "seqs": 1, "heads": 12, "head_dim": 64,
         "length": 701, "window": 0, "ragged": False},
        # a server's running batch of unequal lengths, an e4m3 cache
        {"name": "decode-ragged-e4m3", "kind": "decode", "dtype": "e4m3", "query": "bf16", "seqs": 13, "heads": 12, "head_dim": 64,
         "length": 1500, "window": 0, "ragged": True},
        # the large generation batch
        {"name": "decode-64x4096", "kind": "decode", "dtype": "int8", "query": "bf16", "seqs": 64, "heads": 16, "head_dim": 128,
         "length": 4096, "window": 0, "ragged": False},
        # a few ragged prompts of a floating-point model
        {"name": "context-ragged", "kind": "context", "dtype": "e4m3", "source": "bf16", "seqs": 5, "heads": 12, "head_dim": 64,
         "length": 700, "window": 0, "ragged": True},
        # the 125M-style prefill configuration: a window-64 layer and a full one over 16 fragments of 1024 tokens
        {"name": "prefill-125M-pair", "kind": "prefill", "dtype": "e4m3", "seqs": 16, "heads": 12, "head_dim": 64, "length": 1024,
         "window": 64, "ragged": False, "scales": "rows"},
        # the 1.5B-style prefill configuration: a window-256 layer and a full one over 8 sequences of 4096
        {"name": "prefill-1.5B-pair", "kind": "prefill", "dtype": "e4m3", "seqs": 8, "heads": 16, "head_dim": 128, "length": 4096,
         "window": 256, "ragged": False, "scales": "rows"},
        # one long document
        {"name": "prefill-long", "kind": "prefill", "dtype": "e4m3", "seqs": 1, "heads": 16, "head_dim": 128, "length": 12011,
         "window": 0, "ragged": False, "scales": "rows"},
        # generation for one user with a 125M-style model, calls made one by one
        {"name": "token-one-768", "kind": "token", "seqs": 1, "heads": 12, "head_dim": 64, "length": 300, "graph": False, "ragged": False},
        # generation for 32 users with a 1.5B-style model, a recorded step
        {"name": "token-32-2048", "kind": "token", "seqs": 32, "heads": 16, "head_dim": 128, "length": 2048, "graph": True, "ragged": False},
        # a few short questions to the 1.5B-style model
        {"name": "prompt-short-2048", "kind": "prompt", "seqs": 3, "heads": 16, "head_dim": 128, "length": 200, "window": 0, "ragged": True},
        # the 1.5B-style prompt batch
        {"name": "prompt-32x2048", "kind": "prompt", "seqs": 32, "heads": 16, "head_dim": 128, "length": 2048, "window": 0, "ragged": False},
        # the end of a token step for 32 sequences
        {"name": "head-32", "kind": "head", "rows": 32, "dim": 2048, "vocab": 50257},
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "context", "token", "token", "prompt", "prompt", "head"))
    heads, d = rng.choice(SHAPES)
    width = heads * d
    ragged = rng.random() < 0.5
    if kind == "decode":
        seqs = _log_between(rng, 1, 64)
        return {"kind": kind, "dtype": rng.choice(("int8", "e4m3")), "query": rng.choice(("8bit", "bf16")), "seqs": seqs, "heads": heads,
                "head_dim": d, "length": _log_between(rng, 64, 4096), "window": rng.choice((0, 0, 0, 64, 256)), "ragged": ragged}
    if kind == "prefill":
        length = _log_between(rng, 100, 16384)
        # at most the tokens and the query-key pairs of the largest listed case
        most = max(1, min(32768 // length, int(8 * 4096 ** 2 * 2048 / (length ** 2 * width))))
        return {"kind": kind, "dtype": rng.choice(("e4m3", "e4m3", "int8")), "seqs": _log_between(rng, 1, most), "heads": heads, "head_dim": d,
                "length": min(length, int(4096 * math.sqrt(8 * 2048 / width))), "window": rng.choice((0, 64, 256)), "ragged": ragged,
                "scales": rng.choice(("rows", "rows", "constant"))}
    if kind == "context":
        length = _log_between(rng, 60, 2048)
        return {"kind": kind, "dtype": rng.choice(("int8", "e4m3")), "source": rng.choice(("bf16", "f32")), "seqs": _log_between(rng, 1, max(1, 8192 // length)),
                "heads": heads, "head_dim": d, "length": length, "window": rng.choice((0, 64)), "ragged": ragged}
    if kind == "token":
        return {"kind": kind, "seqs": _log_between(rng, 1, 32), "heads": heads, "head_dim": d, "length": _log_between(rng, 64, 2048),
                "graph": rng.random() < 0.5, "ragged": ragged}
    if kind == "prompt":
        length = _log_between(rng, 40, 2048)
        return {"kind": kind, "seqs": _log_between(rng, 1, max(1, min(32, 32768 // length))), "heads": heads, "head_dim": d, "length": length,
                "window": rng.choice((0, 64)), "ragged": ragged}
    return {"kind": kind, "rows": _log_between(rng, 1, 32), "dim": rng.choice((512, 768, 1024, 1536, 2048)), "vocab": _log_between(rng, 256, 50257)}


def _lengths(case):
    """Tokens of each sequence: `length`, or for a ragged batch anything from a third of it to all of it."""
    n, top = case["seqs"], case["length"]
    if not case["ragged"]:
        return [top] * n
    rng = random.Random(n * 100003 + top)
    return [rng.randint(max(1, top // 3), top) for _ in range(n)]


def _windows(case):
    """(attention width, slope) of the layers of a prefill, context or prompt case."""
    full = (case["length"], 0.0)
    if not case["window"]:
        return [full]
    short = (case["window"], SHORT_SLOPE)
    return [short, full] if case["kind"] == "prefill" else [short]


def _pairs(lengths, window):
    """Query-key pairs of causal self-excluding attention: row t of a sequence sees min(t, window) keys."""
    return sum(s * (s - 1) // 2 if s <= window else window * (window + 1) // 2 + (s - 1 - window) * window for s in lengths)


def _rows(g, n, width, dtype=torch.float32):
    return torch.randn((n, width), device="cuda", generator=g, dtype=dtype)


def _int8(g, shape, rms):
    """int8 values of about that root mean square, as bytes: what conversion of a normal matrix or a normalised row leaves."""
    x = torch.randn(shape, device="cuda", generator=g)
    return x.mul_(rms).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _offsets(lengths):
    return _int32(np.concatenate([[0], np.cumsum(lengths)]))


def _context(case):
    return AttentionContext(0, max_seqs=max(1, case.get("seqs", 1)), max_heads=case.get("heads", 1), max_head_dim=case.get("head_dim", 128))


def _cache(ctx, dtype, case, room, g, filled, key_scale):
    """A cache with `room` rows per sequence, the first `filled` of them from earlier tokens."""
    c = KVCache(ctx, dtype, case["seqs"], case["heads"], room, case["head_dim"])
    if filled:
        shape = (case["seqs"], case["heads"], filled, case["head_dim"])
        if dtype == capi.I8:
            c.k[:, :, :filled] = _int8(g, shape, 24)
            c.v[:, :, :filled] = _int8(g, shape, 24)
        else:
            for plane in (c.k, c.v):
                x = torch.randn(shape, device="cuda", generator=g).mul_(90).clamp_(-448, 448)
                plane[:, :, :filled] = x.to(torch.float8_e4m3fn).view(torch.uint8)
        unit = 1.0 / 24 if dtype == capi.I8 else 1.0 / 90
        c.k_scale[:, :, :filled] = (torch.rand(shape[:3], device="cuda", generator=g) + 0.5) * (key_scale if key_scale else unit)
        c.v_scale[:, :, :filled] = (torch.rand(shape[:3], device="cuda", generator=g) + 0.5) * unit
    return c


def _layer(g, case, width, slope):
    """One int8 layer with matrices as a random model's conversion leaves them: int8 of rms 32, one scale per matrix."""
    dim = qsum = case["heads"] * case["head_dim"]
    return {"proj": _int8(g, (4 * qsum, dim), 32), "combiner": _int8(g, (dim, 4 * qsum), 32), "expand": _int8(g, (qsum, dim), 32),
            "contract": _int8(g, (dim, qsum), 32), "qv_scale": 0.5 / 32, "combiner_scale": 0.5 / 32, "contract_scale": 0.5 / 32,
            "width": width, "slope": slope}


# ---- preparation ---------------------------------------------------------------------------------------------------
def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
    s = {"case": case, "ctx": _context(case)}
    PREPARE[case["kind"]](s, case, g, int(seed))
    return s


def _prepare_decode(s, case, g, seed):
    B, H, d, L = case["seqs"], case["heads"], case["head_dim"], case["length"]
    dtype = DTYPES[case["dtype"]]
    s["cache"] = _cache(s["ctx"], dtype, case, L, g, L, None)
    s["cache"].cache_len.copy_(_int32(_lengths(case)))
    x = _rows(g, B, H * d)
    if case["query"] == "bf16":
        s["q"], s["q_scale"] = x.to(torch.bfloat16), None
    else:
        q, scale = s["ctx"].quantize_rows(x, H, dtype)
        s["q"], s["q_scale"] = q, scale.t().contiguous()


def _prepare_prefill(s, case, g, seed):
    ctx, H, d = s["ctx"], case["heads"], case["head_dim"]
    dtype, lengths = DTYPES[case["dtype"]], _lengths(case)
    n = sum(lengths)
    off = _offsets(lengths)
    s["layers"] = []
    for width, slope in _windows(case):
        qkv = [ctx.quantize_rows(_rows(g, n, H * d), H, dtype) for _ in range(3)]
        if case["scales"] == "constant":  # one number for all queries and one for all values, as the int8 model passes them
            qkv[0], qkv[2] = (qkv[0][0], 0.03 if dtype == capi.I8 else 0.012), (qkv[2][0], 0.03 if dtype == capi.I8 else 0.012)
        spans = ctx.build_spans(off, n, width)
        s["layers"].append({"qkv": qkv, "spans": spans, "tiles": ctx.build_span_tiles(*spans), "slope": slope,
                            "hint": min(width, case["length"]),
                            "period": case["length"] if not case["ragged"] and width >= case["length"] else 0})


def _prepare_context(s, case, g, seed):
    H, d, lengths = case["heads"], case["head_dim"], _lengths(case)
    kind = torch.bfloat16 if case["source"] == "bf16" else torch.float32
    s["qkv"] = [_rows(g, sum(lengths), H * d).to(kind) for _ in range(3)]
    s["offsets"] = _offsets(lengths)
    s["cache"] = _cache(s["ctx"], DTYPES[case["dtype"]], case, case["length"] + 64, g, 0, None)


def _prepare_token(s, case, g, seed):
    ctx, B, H, d, L = s["ctx"], case["seqs"], case["heads"], case["head_dim"], case["length"]
    dim = H * d
    s["layers"] = [_layer(g, case, *((SHORT_WINDOW, SHORT_SLOPE) if i % 2 == 0 else (L + 64, 0.0))) for i in range(LAYERS)]
    s["lengths"] = _int32(_lengths(case))
    s["start"] = s["lengths"].repeat(LAYERS, 1)
    lens = s["lens"] = s["start"].clone()
    s["caches"] = []
    for i in range(LAYERS):
        c = _cache(ctx, capi.I8, case, L + 64, g, L, 0.02)
        c.v_scale.fill_(VEC_SCALE)
        c.cache_len = lens[i]
        s["caches"].append(c)
    s["rope"] = ctx.fill_rope_table(d, L + 64)
    s["embed"] = _int8(g, (EMBED_ROWS, dim), 32)
    s["labels"] = torch.randint(0, EMBED_ROWS, (B,), dtype=torch.int32, device="cuda", generator=g)
    s["state"] = torch.empty((B, dim), dtype=torch.float32, device="cuda")
    s["keep"] = {}
    s["graph"] = None
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _token_step(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s["result"] = _token_step(s)
        s["graph"] = graph


def _prepare_prompt(s, case, g, seed):
    ctx, H, d, lengths = s["ctx"], case["heads"], case["head_dim"], _lengths(case)
    n, dim = sum(lengths), H * d
    width, slope = _windows(case)[0]
    s["layer"] = _layer(g, case, width, slope)
    s["cache"] = KVCache(ctx, capi.I8, case["seqs"], H, case["length"] + 64, d)
    s["cache"].v_scale.fill_(VEC_SCALE)
    s["offsets"] = _offsets(lengths)
    s["pos"] = _int32(np.concatenate([np.arange(x) for x in lengths]))
    s["rope"] = ctx.fill_rope_table(d, case["length"] + 64)
    s["spans"] = ctx.build_spans(s["offsets"], n, width)
    s["tiles"] = ctx.build_span_tiles(*s["spans"])
    s["period"] = case["length"] if not case["ragged"] and width >= case["length"] else 0
    s["embed"] = _int8(g, (EMBED_ROWS, dim), 32)
    s["labels"] = torch.randint(0, EMBED_ROWS, (n,), dtype=torch.int32, device="cuda", generator=g)
    s["state"] = torch.empty((n, dim), dtype=torch.float32, device="cuda")


def _prepare_head(s, case, g, seed):
    s["norm"] = _int8(g, (case["rows"], case["dim"]), 24)
    s["final"] = _int8(g, (case["vocab"], case["dim"]), 32)
    s["bias"] = torch.randn(case["vocab"], device="cuda", generator=g) * 0.1
    s["scale"] = math.sqrt(1.0 / case["dim"]) / 0.693147 / 32 * VEC_SCALE
    s["planes"] = torch.empty(16 * case["rows"] * case["vocab"], dtype=torch.int32, device="cuda")
    s["seed"] = seed


PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "context": _prepare_context, "token": _prepare_token,
           "prompt": _prepare_prompt, "head": _prepare_head}


# ---- one pass ------------------------------------------------------------------------------------------------------
def run(state):
    return RUN[state["case"]["kind"]](state)


def _run_decode(s):
    case = s["case"]
    window, slope = (case["window"], SHORT_SLOPE) if case["window"] else (case["length"], 0.0)
    return s["ctx"].compute_val_lookup_decode(s["cache"], s["q"], s["q_scale"], window, slope)


def _run_prefill(s):
    case, outs = s["case"], []
    for layer in s["layers"]:
        (q, qs), (k, ks), (v, vs) = layer["qkv"]
        outs.append(s["ctx"].compute_val_lookup(DTYPES[case["dtype"]], case["heads"], q, k, v, qs, ks, vs, *layer["spans"], layer["slope"],
                                                out_f16=True, causal_period=layer["period"], span_tiles=layer["tiles"], span_len_hint=layer["hint"]))
    return outs


def _run_context(s):
    case, ctx, cache = s["case"], s["ctx"], s["cache"]
    H, dtype, n = case["heads"], DTYPES[case["dtype"]], s["qkv"][0].shape[0]
    width, slope = _windows(case)[0]
    spans = ctx.build_spans(s["offsets"], n, width)
    tiles = ctx.build_span_tiles(*spans)
    (q, qs), (k, ks), (v, vs) = (ctx.quantize_rows(x, H, dtype) for x in s["qkv"])
    out = ctx.compute_val_lookup(dtype, H, q, k, v, qs, ks, vs, *spans, slope, span_tiles=tiles, span_len_hint=min(width, case["length"]))
    cache.cache_len.zero_()  # a new batch
    cache.fill_from_prefill(s["offsets"], k, ks, v, vs)
    return {"out": out, "q": q, "q_scale": qs, "k": cache.k, "v": cache.v, "k_scale": cache.k_scale, "v_scale": cache.v_scale,
            "cache_len": cache.cache_len}


def _token_step(s):
    ctx, state = s["ctx"], s["state"]
    torch.add(s["start"], 0, out=s["lens"])  # the token's place in every cache
    ctx.embed_rows(s["labels"], s["embed"], 1.0 / 32, out=state)
    pending = None
    for layer, cache in zip(s["layers"], s["caches"]):
        _, pending = add_lookup_product(ctx, layer, cache, s["lengths"], s["rope"], state, scratch=s["keep"], pending=pending, defer=True)
    norm = flush_state(ctx, pending, state)
    low, high = min(_lengths(s["case"])), max(_lengths(s["case"])) + 1  # the rows the new tokens went to
    return {"state": state, "norm": norm, "lens": s["lens"], "k": [c.k[:, :, low:high] for c in s["caches"]], "v": [c.v[:, :, low:high] for c in s["caches"]],
            "k_scale": [c.k_scale[:, :, low:high] for c in s["caches"]]}


def _run_token(s):
    if s["graph"] is None:
        return _token_step(s)
    s["graph"].replay()
    return s["result"]


def _run_prompt(s):
    ctx, cache, state = s["ctx"], s["cache"], s["state"]
    ctx.embed_rows(s["labels"], s["embed"], 1.0 / 32, out=state)
    cache.cache_len.zero_()  # new prompts
    _, norm = add_lookup_product_prompt(ctx, s["layer"], cache, s["offsets"], s["pos"], s["rope"], state, *s["spans"], span_tiles=s["tiles"],
                                        causal_period=s["period"], want_norm=True, want_val=False)
    return {"state": state, "norm": norm, "k": cache.k, "v": cache.v, "k_scale": cache.k_scale, "cache_len": cache.cache_len}


def _run_head(s):
    ctx = s["ctx"]
    logits = ctx.matmul_i8(s["norm"], s["final"], mode=capi.MM_I32_PLANES, out=s["planes"])
    prob, best = ctx.softmax_rows(logits, s["scale"], s["bias"])
    choice = ctx.sample_rows(prob, 0.8, seed=s["seed"])
    return {"prob": prob, "best": best, "choice": choice}


RUN = {"decode": _run_decode, "prefill": _run_prefill, "context": _run_context, "token": _run_token, "prompt": _run_prompt, "head": _run_head}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    if case["kind"] == "head":
        m, n, k = case["rows"], case["vocab"], case["dim"]
        return {"bytes": n * k + m * k + 4 * n + 4 * m * n + 8 * m, "flops": 2 * m * n * k}
    H, d, lengths = case["heads"], case["head_dim"], _lengths(case)
    width, tokens = H * d, sum(lengths)
    if case["kind"] == "decode":
        window = case["window"] or case["length"]
        keys = sum(min(x - 1, window) for x in lengths)
        q = 2 * width if case["query"] == "bf16" else width + 4 * H
        return {"bytes": keys * H * (2 * d + 8) + case["seqs"] * (q + 4 * width + 4), "flops": 4 * keys * width}
    if case["kind"] == "prefill":
        scales = (1 if case["scales"] == "constant" else 3) * 4 * H
        layers = _windows(case)
        return {"bytes": len(layers) * tokens * (3 * width + scales + 2 * width + 8), "flops": sum(4 * width * _pairs(lengths, w) for w, _ in layers)}
    if case["kind"] == "context":
        source = 2 if case["source"] == "bf16" else 4
        # in: Q, K, V; out: attention, the quantised queries and the cache's rows with their scales
        return {"bytes": tokens * (3 * source * width + 4 * width + 3 * width + 12 * H), "flops": 4 * width * _pairs(lengths, _windows(case)[0][0])}
    matrices = 10 * width * width  # projections 4, combiner 4, expand 1, contract 1
    if case["kind"] == "token":
        keys = sum(min(x, SHORT_WINDOW) + x for x in lengths) * (LAYERS // 2)
        return {"bytes": LAYERS * (matrices + case["seqs"] * H * (2 * d + 8)) + keys * H * (2 * d + 8) + case["seqs"] * (width + 5 * width + 4 * d),
                "flops": LAYERS * 2 * matrices * case["seqs"] + 4 * keys * width}
    # prompt: embedding rows in, matrices in, state and its normalisation out, the cache's rows out
    return {"bytes": matrices + tokens * (width + 5 * width + 2 * width + 4 * H + 4 * d), "flops": 2 * matrices * tokens + 4 * width * _pairs(lengths, _windows(case)[0][0])}


def tolerance(case):
    if case["kind"] == "decode":  # 8-bit inputs, everything behind them in 32 bits
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "head":    # exact sums of int8 products, the softmax in 32 bits
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] in ("prefill", "context"):  # weights and scaled values in 16 bits; quantised rows are exact
        return {"rel": 2e-3, "max": 2e-2}
    # the layer rounds to int8 behind every step: a value on the edge goes to its other neighbour with the last bit of a
    # sum, and the values computed from it move by its share
    return {"rel": 5e-3, "max": 0.1, "differ": 5e-3}
