"""What this library is timed on: the calls a program that serves a quantised
model makes, through the entry points it makes them with.

Weights are GGML K-quant blocks of Gaussian rows (sigma 0.02), quantised by
ggml's reference quantisers; activations are N(0, 1) in 16 bits; KV caches
are N(0, 1) in fp16, or int8 with per-(position, KV head) scales.  Every call
has inputs of its own (no call feeds the next), so each output has the error
of one call.

Layers go through the C++ API (reflex::infer::*), their argument blocks built
once, as a runtime builds them when it lays out a model; single products, the
batched gather and the bf16 products (these two are not in the C++ API)
through the Python binding of the C ABI.  A decode step is captured once into
a HIP graph and replayed, as serving loops do and as bench.py does; every
other pass issues its calls on the current stream.

Kinds of case:
  gemv    one matrix and one token: a single projection, the LM head
  decode  one token through `layers` decoder layers: fused Q/K/V triple,
          attention over `ctx` positions (none if 0), output projection with
          residual, gate+up pair, down projection with residual
  linear  `tokens` tokens through one layer's matrices, one call per matrix:
          "layer" is q, k, v, o, gate, up and down, "mlp" the last three
  embed   a prompt's embedding rows, Zipf(1.1) ids
  attn    attention of one layer; `tokens` 0 is one decode token over `start`
          positions, otherwise a prompt of `tokens` after `start` cached ones
"mix" is the layout of common 4-bit files: v, down (and nothing else) in
Q6_K, the rest in `type`.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "reflex-infer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import rxq4  # noqa: E402
from rxq4 import api, capi  # noqa: E402

DEV = "cuda:0"
BYTES = {12: 144, 13: 176, 14: 210}  # per 256 weights: Q4_K, Q5_K, Q6_K


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one projection of a small model, fp32 out: the smallest call, launch latency
        {"name": "projection_2048", "kind": "gemv", "type": 12, "M": 2048, "K": 2048, "out": "f32"},
        # a decode step of a 3B-class model's projections (bench.py's layer set)
        {"name": "decode_2048", "kind": "decode", "type": 12, "mix": False, "hidden": 2048, "ffn": 11008,
         "heads": 16, "kv": 2, "head_dim": 128, "layers": 12, "ctx": 0},
        # a decode step of a 13B-class model in the mixed file layout, 2000 tokens in
        {"name": "decode_5120_mix", "kind": "decode", "type": 12, "mix": True, "hidden": 5120, "ffn": 13824,
         "heads": 40, "kv": 8, "head_dim": 128, "layers": 4, "ctx": 2000},
        # the logits of one token: the vocabulary's matrix is Q6_K in mixed files
        {"name": "lm_head_q6k", "kind": "gemv", "type": 14, "M": 151936, "K": 2048, "out": "f32"},
        # a long prompt's embedding rows
        {"name": "embed_4096", "kind": "embed", "type": 12, "vocab": 151936, "hidden": 2048, "tokens": 4096},
        # eight sequences decoding together
        {"name": "batch_8", "kind": "linear", "part": "layer", "type": 12, "mix": True, "dtype": "f16", "tokens": 8,
         "hidden": 2048, "ffn": 11008, "heads": 16, "kv": 2, "head_dim": 128},
        # a short prompt (or a draft being checked, or 45 sequences), odd length
        {"name": "prompt_45", "kind": "linear", "part": "layer", "type": 12, "mix": True, "dtype": "f16", "tokens": 45,
         "hidden": 2048, "ffn": 11008, "heads": 16, "kv": 2, "head_dim": 128},
        # a prompt of the usual prefill chunk, bf16 (bench.py's prefill shapes)
        {"name": "prefill_512_bf16", "kind": "linear", "part": "mlp", "type": 12, "mix": False, "dtype": "bf16",
         "tokens": 512, "hidden": 2048, "ffn": 11008, "heads": 16, "kv": 2, "head_dim": 128},
        # a long prompt through an 8B-class layer, mixed file layout: the largest
        {"name": "prefill_2048_mix", "kind": "linear", "part": "layer", "type": 12, "mix": True, "dtype": "f16",
         "tokens": 2048, "hidden": 4096, "ffn": 14336, "heads": 32, "kv": 8, "head_dim": 128},
        # decode attention over a long int8 cache
        {"name": "attn_decode_16k_int8", "kind": "attn", "tokens": 0, "start": 16000, "heads": 32, "kv": 8,
         "head_dim": 128, "int8": True},
        # a long prompt's attention from an empty cache
        {"name": "attn_prefill_2048", "kind": "attn", "tokens": 2048, "start": 0, "heads": 32, "kv": 8,
         "head_dim": 128, "int8": False},
        # the next turn of a chat: a short message after 8000 cached positions
        {"name": "attn_turn_45_8k", "kind": "attn", "tokens": 45, "start": 8000, "heads": 32, "kv": 8,
         "head_dim": 128, "int8": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng, wide):
    """heads, kv, head_dim; `wide` also the head sizes other than 64 and 128."""
    hd = rng.choice([128, 128, 128, 128, 64, 64] + ([80, 96, 256] if wide else []))
    kv = rng.choice([1, 2, 4, 8, 8, 16])
    return kv * rng.choice([1, 2, 4, 4, 5, 7, 8]), kv, hd


def _ragged(rows, K, tokens=1):
    """Whether a Q4_K product of one to three tokens leaves waves of its last
    workgroup without rows.  The first build that these cases were run on read
    past the matrix there (its row kernel for long rows deals whole rows to
    waves, four waves to a workgroup), so that such sizes cannot be run on it."""
    slots, total = K // 64, sum(rows)
    if slots <= 64 and 64 % slots == 0:
        return False
    wave = -(-total // 2048) * (K // 256) * 144
    if wave <= 16384 and 8 * (8192 if wave <= 8192 else 16384) + 144 * slots * tokens <= 160 << 10:
        return False
    per = -(-total // 1024)
    return sum(-(-r // per) for r in rows) % 4 != 0


def draw(rng):
    while True:
        c = _draw(rng)
        if c["kind"] == "gemv":
            products = [([c["M"]], c["K"])] if c["type"] == 12 else []
        elif c["kind"] == "decode":
            H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv"] * c["head_dim"]
            products = [([H], Q), ([F, F], H)] + ([] if c["mix"] else [([Q, KV, KV], H), ([H], F)])
            products = products if c["type"] == 12 else []
        elif c["kind"] == "linear" and c["tokens"] < 4 and c["dtype"] == "f16":
            products = [([M], K) for _, M, K, t in _matrices(c) if t == 12]
        else:
            products = []
        if not any(_ragged(rows, K, c.get("tokens", 1)) for rows, K in products):
            return c


def _draw(rng):
    kind = rng.choice(["gemv", "decode", "linear", "linear", "linear", "embed", "attn", "attn", "attn"])
    typ = rng.choice([12, 12, 12, 13, 14])
    if kind == "gemv":
        K = 256 * _log(rng, 2, 56)
        return {"kind": kind, "type": typ, "M": _log(rng, 256, min(152064, (320 << 20) // K)), "K": K,
                "out": rng.choice(["f32", "f16", "add"])}
    if kind == "embed":
        hidden = 256 * _log(rng, 3, 20)
        return {"kind": kind, "type": rng.choice([12, 14]), "vocab": _log(rng, 32000, 152000 * 2048 // max(hidden, 2048)),
                "hidden": hidden, "tokens": _log(rng, 1, 8192)}
    if kind == "attn":
        heads, kv, hd = _heads(rng, True)
        while heads > 64:
            heads, kv, hd = _heads(rng, True)
        tokens = 0 if rng.random() < 0.4 else _log(rng, 2, 2048)
        start = _log(rng, 256, 32768) if tokens == 0 else rng.choice([0, _log(rng, 16, 16384), _log(rng, 16, 16384)])
        # no more work than a prompt of 2048 tokens for 32 heads of 128 (a
        # tenth of it for the head sizes that few models have)
        most = (1 << 33) * (1.0 if hd in (64, 128) else 0.1)
        while tokens and heads * hd * tokens * (start + tokens / 2) > most:
            tokens, start = (tokens + 1) // 2, start // 2
        return {"kind": kind, "tokens": tokens, "start": start, "heads": heads, "kv": kv, "head_dim": hd,
                "int8": rng.random() < 0.3}
    hd = rng.choice([64, 128, 128])
    hidden = 256 * _log(rng, 4, 20)
    heads = hidden // hd
    kv = rng.choice([k for k in (1, 2, 4, 5, 6, 8, 10, 16) if heads % k == 0 and k * hd <= hidden])
    ffn = 256 * int(hidden * rng.uniform(2.5, 5.5) / 256)
    case = {"kind": kind, "type": 13 if typ == 13 else 12, "mix": typ != 12, "hidden": hidden, "ffn": ffn,
            "heads": heads, "kv": kv, "head_dim": hd}
    if kind == "decode":
        layer = sum(M * K for _, M, K, _ in _matrices(case)) * 160 // 256
        return dict(case, layers=max(2, min(12, (300 << 20) // layer)), ctx=rng.choice([0, _log(rng, 1, 8192), _log(rng, 64, 8192)]))
    tokens = _log(rng, 2, 2048)
    part = rng.choice(["layer", "mlp"])
    most = sum(M * K for _, M, K, _ in _matrices(listed()[8])) * 2048
    while tokens * sum(M * K for _, M, K, _ in _matrices(case)) > most:
        tokens = (tokens + 1) // 2
    return dict(case, part=part, tokens=tokens, dtype=rng.choice(["f16", "f16", "bf16"]))


def _matrices(c):
    """(name, rows, row length, type) of a layer's matrices."""
    H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv"] * c["head_dim"]
    t, t6 = c["type"], 14 if c["mix"] else c["type"]
    mlp = [("gate", F, H, t), ("up", F, H, t), ("down", H, F, t6)]
    if c.get("part") == "mlp":
        return mlp
    return [("q", Q, H, t), ("k", KV, H, t), ("v", KV, H, t6), ("o", H, Q, t)] + mlp


# ------------------------------------------------------------------- inputs
class _Gen:
    """The case's random inputs, in one order whatever is kept of them."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.g, device=DEV)

    def weights(self, M, K, t):
        return capi.quantize_ggml(self.normal(M, K).mul_(0.02), t)

    def x(self, *shape, bf16=False):
        return self.normal(*shape).to(torch.bfloat16 if bf16 else torch.float16)

    def cache(self, c, n):
        """K, V and their scales (None for fp16)."""
        shape = (n, c["kv"], c["head_dim"])
        if not c.get("int8"):
            return self.x(*shape), self.x(*shape), None, None
        k, v = (self.normal(*shape).mul_(40).round_().clamp_(-127, 127).to(torch.int8) for _ in range(2))
        ks, vs = (self.uniform(n, c["kv"]).mul_(0.01).add_(0.02) for _ in range(2))
        return k, v, ks, vs


def _inputs(c, seed):
    g, kind = _Gen(seed), c["kind"]
    if kind == "gemv":
        d = {"w": g.weights(c["M"], c["K"], c["type"]), "x": g.x(c["K"])}
        if c["out"] == "add":
            d["res"] = g.x(c["M"])
        return d
    if kind == "embed":
        w = g.weights(c["vocab"], c["hidden"], c["type"])
        p = torch.arange(1, c["vocab"] + 1, device=DEV, dtype=torch.float64).pow_(-1.1).cumsum_(0)
        ranks = torch.searchsorted(p, g.uniform(c["tokens"]).double() * p[-1]).clamp_(max=c["vocab"] - 1)
        order = torch.argsort(g.uniform(c["vocab"]))  # a frequent word's row is anywhere in the table
        return {"w": w, "ids": order[ranks].to(torch.int32)}
    if kind == "attn":
        n = c["start"] + c["tokens"]
        k, v, ks, vs = g.cache(c, n)
        return {"q": g.x(max(1, c["tokens"]), c["heads"] * c["head_dim"]), "k": k, "v": v, "ks": ks, "vs": vs}
    if kind == "linear":
        bf16 = c["dtype"] == "bf16"
        ms = _matrices(c)
        return {"w": [g.weights(M, K, t) for _, M, K, t in ms],
                "x": {K: g.x(c["tokens"], K, bf16=bf16) for K in sorted({K for _, _, K, _ in ms})}}
    layers = []
    for _ in range(c["layers"]):
        d = {name: g.weights(M, K, t) for name, M, K, t in _matrices(c)}
        d["x"], d["xo"], d["x2"], d["xd"] = (g.x(n) for n in (c["hidden"], c["heads"] * c["head_dim"], c["hidden"], c["ffn"]))
        d["res"], d["res2"] = g.x(c["hidden"]), g.x(c["hidden"])
        if c["ctx"]:
            d["kc"], d["vc"], _, _ = g.cache(c, c["ctx"])
            d["qa"] = g.x(c["heads"] * c["head_dim"])
        layers.append(d)
    return {"layers": layers}


# --------------------------------------------------------------------- a pass
def _call(name, args):
    status = api.call(name, args)
    if status != rxq4.SUCCESS:
        raise rxq4.RxQ4Error(status, name)


def _half(*shape, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _attention(out, q, k, v, c, tokens, start, stream, ks=None, vs=None):
    H, G, D = c["heads"], c["kv"], c["head_dim"]
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    tail = (float(D) ** -0.5, ks is not None, p(ks), p(vs), stream)
    if tokens == 0:
        return ("flash_attention_decode", api.AttentionDecodeArgs(p(out), p(q), p(k), p(v), H, G, D, start, *tail))
    return ("flash_attention_prefill_batched",
            api.AttentionPrefillBatchedArgs(p(out), p(q), p(k), p(v), H, G, D, tokens, start, *tail))


def _decode_calls(c, s, stream):
    """The calls of a decode step and its outputs, a row per layer."""
    H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv"] * c["head_dim"]
    L, t, t6 = c["layers"], c["type"], 14 if c["mix"] else c["type"]
    out = {"qkv": _half(L, Q + 2 * KV), "o": _half(L, H), "gate_up": _half(L, 2 * F), "down": _half(L, H)}
    if c["ctx"]:
        out["attn"] = _half(L, Q)
    calls = []
    for i, d in enumerate(s["layers"]):
        p = {n: (v.data_ptr() if v is not None else None) for n, v in d.items()}
        y = [out["qkv"][i, a:].data_ptr() for a in (0, Q, Q + KV)]
        calls.append(("gemv_quant_triple", api.GemvQuantTripleArgs(
            y[0], p["q"], p["q"], t, Q, y[1], p["k"], p["k"], t, KV, y[2], p["v"], p["v"], t6, KV, p["x"], H, stream)))
        if c["ctx"]:
            calls.append(_attention(out["attn"][i], d["qa"], d["kc"], d["vc"], c, 0, c["ctx"], stream))
        calls.append(("gemv_quant_add", api.GemvQuantAddArgs(
            out["o"][i].data_ptr(), p["o"], p["o"], t, p["xo"], p["res"], H, Q, stream)))
        calls.append(("gemv_quant_pair", api.GemvQuantPairArgs(
            out["gate_up"][i].data_ptr(), p["gate"], p["gate"], t, F, out["gate_up"][i, F:].data_ptr(),
            p["up"], p["up"], t, F, p["x2"], H, stream)))
        calls.append(("gemv_quant_add", api.GemvQuantAddArgs(
            out["down"][i].data_ptr(), p["down"], p["down"], t6, p["xd"], p["res2"], H, F, stream)))
    return calls, out


def prepare(case, seed):
    rxq4.load()
    s = _inputs(case, seed)
    kind = case["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "gemv":
        return {"case": case, "in": s, "out": _half(case["M"], dtype=torch.float32 if case["out"] == "f32" else torch.float16)}
    if kind == "attn":
        out = torch.empty_like(s["q"])
        call = _attention(out, s["q"], s["k"], s["v"], case, case["tokens"], case["start"], stream, s["ks"], s["vs"])
        return {"case": case, "in": s, "calls": [call], "out": out}
    if kind == "embed":
        return {"case": case, "in": s, "out": _half(case["tokens"], case["hidden"])}
    if kind == "linear":
        N, dt = case["tokens"], torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        ms = _matrices(case)
        out = {n: _half(N, M, dtype=dt) for n, M, _, _ in ms}
        if case["dtype"] == "bf16":
            return {"case": case, "in": s, "ms": [(out[n], w, s["x"][K], M, N, K, t) for (n, M, K, t), w in zip(ms, s["w"])], "out": out}
        calls = [("gemm_quant_batched", api.GemmQuantBatchedArgs(
            out[n].data_ptr(), w.data_ptr(), w.data_ptr(), t, s["x"][K].data_ptr(), M, N, K, stream))
            for (n, M, K, t), w in zip(ms, s["w"])]
        return {"case": case, "in": s, "calls": calls, "out": out}
    # a decode step: one eager pass on the side stream, then its capture
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    calls, out = _decode_calls(case, s, side.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        for name, args in calls:
            _call(name, args)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side, capture_error_mode="relaxed"):
        for name, args in calls:
            _call(name, args)
    return {"case": case, "in": s, "graph": graph, "side": side, "out": out}


def run(state):
    if "graph" in state:
        state["graph"].replay()
    elif "calls" in state:
        for name, args in state["calls"]:
            _call(name, args)
    elif "ms" in state:
        for y, w, x, M, N, K, t in state["ms"]:
            capi.gemm(y, w, x, M, N, K, ggml_type=t)
    else:
        c, s, y = state["case"], state["in"], state["out"]
        if c["kind"] == "embed":
            capi.embed_rows_f16(y, s["w"], c["vocab"], s["ids"], c["hidden"], ggml_type=c["type"])
        elif c["out"] == "f32":
            capi.gemv_f32(y, s["w"], s["x"], c["M"], c["K"], ggml_type=c["type"])
        elif c["out"] == "f16":
            capi.gemv_f16(y, s["w"], s["x"], c["M"], c["K"], ggml_type=c["type"])
        else:
            capi.gemv_add_f16(y, s["w"], s["x"], s["res"], c["M"], c["K"], ggml_type=c["type"])
    return state["out"]


# --------------------------------------------------- work, tolerance, 64 bits
def _attn_work(c, tokens, start):
    H, G, D = c["heads"], c["kv"], c["head_dim"]
    n, N = start + tokens, max(1, tokens)
    pairs = start if tokens == 0 else tokens * start + tokens * (tokens + 1) / 2
    cache = 2 * n * G * (D + 4 if c.get("int8") else 2 * D)
    return cache + 4 * N * H * D, 4 * H * D * pairs


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        y = {"f32": 4, "f16": 2, "add": 4}[c["out"]]
        return {"bytes": c["M"] * c["K"] // 256 * BYTES[c["type"]] + 2 * c["K"] + y * c["M"], "flops": 2 * c["M"] * c["K"]}
    if kind == "embed":
        # rows that Zipf(1.1) ids name, on average
        V, n = c["vocab"], c["tokens"]
        p = torch.arange(1, V + 1, dtype=torch.float64).pow_(-1.1)
        rows = float((1 - (1 - p / p.sum()).pow(n)).sum())
        H = c["hidden"]
        return {"bytes": rows * H // 256 * BYTES[c["type"]] + 2 * n * H + 4 * n, "flops": 2 * n * H}
    if kind == "attn":
        b, f = _attn_work(c, c["tokens"], c["start"])
        return {"bytes": b, "flops": f}
    ms = _matrices(c)
    w = sum(M * K // 256 * BYTES[t] for _, M, K, t in ms)
    mk = sum(M * K for _, M, K, _ in ms)
    if kind == "linear":
        N = c["tokens"]
        return {"bytes": w + 2 * N * (sum({K for _, _, K, _ in ms}) + sum(M for _, M, _, _ in ms)), "flops": 2 * N * mk}
    H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv"] * c["head_dim"]
    b, f = w + 2 * (2 * H + Q + F) + 2 * (Q + 2 * KV + 2 * F + 4 * H), 2 * mk
    if c["ctx"]:
        ab, af = _attn_work(c, 0, c["ctx"])
        b, f = b + ab, f + af
    return {"bytes": c["layers"] * b, "flops": c["layers"] * f}


def tolerance(case):
    # four times the distance from exact() that was measured over draw()'s ranges
    if case["kind"] == "embed":
        return "exact"  # one product and one subtraction, then one rounding: bit for bit
    if case["kind"] == "gemv" and case["out"] == "f32":
        return {"rel": 4e-5}  # 1e-5: fp32 sums of products with 1024 + q, the 1024 taken off as a sum
    if case.get("dtype") == "bf16":
        return {"rel": 9e-3}  # 2.3e-3: weights rounded to bf16, bf16 outputs
    return {"rel": 1.2e-3}    # 3e-4: fp16 outputs (and weights, in the matrix-core products)


def _dequant(w, M, K, t, lo=0, hi=None):
    """Rows [lo, hi) of the blocks `w` in float64, from the format's definition."""
    hi = M if hi is None else hi
    b = w.reshape(M, -1)[lo:hi].reshape(-1, BYTES[t])
    f16 = lambda a, o: a[:, o:o + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if t == 14:
        ql, qh = b[:, :128].reshape(-1, 2, 64).int(), b[:, 128:192].reshape(-1, 2, 32).int()
        sc, d = b[:, 192:208].contiguous().view(torch.int8).double(), f16(b, 208)
        q = torch.stack([(ql[:, :, :32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 32:] >> 4) | ((qh >> 6) << 4)], 2)
        v = (q.reshape(-1, 16, 16) - 32).double() * (d * sc)[:, :, None]
        return v.reshape(hi - lo, K)
    d, dmin, s = f16(b, 0), f16(b, 2), b[:, 4:16].int()
    lo6, hi6 = s[:, :8], s[:, 8:12]
    sc = torch.cat([lo6[:, :4] & 63, (hi6 & 15) | ((lo6[:, :4] >> 6) << 4)], 1)
    mn = torch.cat([lo6[:, 4:] & 63, (hi6 >> 4) | ((lo6[:, 4:] >> 6) << 4)], 1)
    qs = b[:, BYTES[t] - 128:].reshape(-1, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if t == 13:
        bit = torch.arange(8, device=w.device, dtype=torch.int32)[None, :, None]
        q = q | (((b[:, 16:48].int()[:, None, :] >> bit) & 1) << 4)
    v = (d * sc.double())[:, :, None] * q.double() - (dmin * mn.double())[:, :, None]
    return v.reshape(hi - lo, K)


def _product(w, x, M, K, t):
    """x [N x K] times the rows of w, in float64, some rows at a time."""
    step = max(1, (64 << 20) // K)
    return torch.cat([x.double() @ _dequant(w, M, K, t, a, min(M, a + step)).t().contiguous()
                      for a in range(0, M, step)], 1)


def _attention64(c, q, k, v, tokens, start, ks=None, vs=None):
    H, G, D = c["heads"], c["kv"], c["head_dim"]
    N, n = max(1, tokens), start + tokens
    out = torch.empty(N, H, D, dtype=torch.float64, device=q.device)
    q = q.double().view(N, H, D)
    for g in range(G):
        kk, vv = k[:, g].double(), v[:, g].double()
        if ks is not None:
            kk, vv = kk * ks[:, g, None].double(), vv * vs[:, g, None].double()
        kt = kk.t().contiguous()
        for h in range(g * (H // G), (g + 1) * (H // G)):
            for a in range(0, N, 512):
                s = (q[a:a + 512, h].contiguous() @ kt) * float(D) ** -0.5
                if tokens:
                    pos = torch.arange(n, device=q.device)[None, :]
                    s.masked_fill_(pos > start + a + torch.arange(s.shape[0], device=q.device)[:, None], -math.inf)
                out[a:a + 512, h] = torch.softmax(s, 1) @ vv
    return out.reshape(N, H * D)


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    if c["kind"] == "gemv":
        y = _product(s["w"], s["x"][None], c["M"], c["K"], c["type"])[0]
        return y + s["res"].double() if c["out"] == "add" else y
    if c["kind"] == "embed":
        return _dequant(s["w"].view(c["vocab"], -1)[s["ids"].long()], c["tokens"], c["hidden"], c["type"])
    if c["kind"] == "attn":
        return _attention64(c, s["q"], s["k"], s["v"], c["tokens"], c["start"], s["ks"], s["vs"])
    if c["kind"] == "linear":
        return {n: _product(w, s["x"][K], M, K, t) for (n, M, K, t), w in zip(_matrices(c), s["w"])}
    rows = {"qkv": [], "o": [], "gate_up": [], "down": []}
    if c["ctx"]:
        rows["attn"] = []
    for d in s["layers"]:
        y = {n: _product(d[n], d[{"o": "xo", "gate": "x2", "up": "x2", "down": "xd"}.get(n, "x")][None], M, K, t)[0]
             for n, M, K, t in _matrices(c)}
        rows["qkv"].append(torch.cat([y["q"], y["k"], y["v"]]))
        rows["o"].append(y["o"] + d["res"].double())
        rows["gate_up"].append(torch.cat([y["gate"], y["up"]]))
        rows["down"].append(y["down"] + d["res2"].double())
        if c["ctx"]:
            rows["attn"].append(_attention64(c, d["qa"][None], d["kc"], d["vc"], 0, c["ctx"])[0])
    return {n: torch.stack(v) for n, v in rows.items()}
