"""The work that programs have this library do, as measurable cases.

Every case is one stretch of a transformer forward pass through the public
entry points of ``rustllm_amd.abi`` (the binding of the C ABI): a decode
step, a decoder layer's prefill, the attention core in its forms, the
reference's separate score calls, normalisation, element-wise work and the
embedding.  Projections are not part of the library, so the rows that a
projection would produce are inputs.

``listed()`` holds named cases, ``draw(rng)`` gives more of the same ranges.
``prepare`` makes the device tensors a program has in hand before the call,
``run`` is one pass, ``exact`` the same outputs in 64 bits from plain torch,
``work`` the bytes and operations no implementation can do without.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from rustllm_amd import abi

EPS = 1e-5
THETA = 10000.0

# (query heads, KV heads): the head groupings of the test suite and the benchmark.
HEADS = [(9, 3), (15, 5), (32, 8), (8, 8), (12, 3)]
# (hidden, query heads, KV heads, FFN) of whole layers, head size 64.
LAYERS = [(576, 9, 3, 1536), (960, 15, 5, 2560)]
DTYPES = {"f16": (torch.float16, np.float16, 2), "f32": (torch.float32, np.float32, 4)}

_context: abi.Context | None = None


def context() -> abi.Context:
    """The process's one context, as a program on one GPU holds it."""
    global _context
    if _context is None:
        _context = abi.Context(0)
    return _context


def listed() -> list[dict]:
    return [
        # One token through a layer's non-projection work, half-full cache: six small launches.
        {"name": "decode_step_f16", "kind": "decode_step", "dtype": "f16", "layer": 1,
         "cached": 1535, "capacity": 4096},
        # Attention of several sequences decoding together, each over a long ragged cache.
        {"name": "decode_batch_f16", "kind": "attention", "dtype": "f16", "batch": 8, "heads": 15,
         "kv_heads": 5, "head_dim": 64, "queries": 1, "cached": 3000, "capacity": 4096},
        # A 4096-token prompt through a layer's non-projection chain with the scores in memory,
        # as the reference composes it (the benchmark's headline chain).
        {"name": "prefill_layer_f16", "kind": "prefill_layer", "dtype": "f16", "layer": 1,
         "tokens": 4096},
        # The fused attention core over the same prompt.
        {"name": "prefill_attention_f16", "kind": "attention", "dtype": "f16", "batch": 1,
         "heads": 15, "kv_heads": 5, "head_dim": 64, "queries": 4096, "cached": 0,
         "capacity": 4096},
        # The same in f32 (models loaded without conversion), a ragged prompt.
        {"name": "prefill_attention_f32", "kind": "attention", "dtype": "f32", "batch": 1,
         "heads": 15, "kv_heads": 5, "head_dim": 64, "queries": 3001, "cached": 0,
         "capacity": 4096},
        # A prompt taken in chunks: new tokens after cached ones, heads of 128.
        {"name": "chunked_prefill_f16", "kind": "attention", "dtype": "f16", "batch": 1,
         "heads": 32, "kv_heads": 8, "head_dim": 128, "queries": 512, "cached": 3000,
         "capacity": 4096},
        # A prompt of a model whose head size is not a multiple of 32.
        {"name": "head80_prefill_f16", "kind": "attention", "dtype": "f16", "batch": 1,
         "heads": 8, "kv_heads": 8, "head_dim": 80, "queries": 1021, "cached": 0,
         "capacity": 1024},
        # The reference's three attention calls (scores, scale/mask + softmax, values), odd length.
        {"name": "score_calls_f16", "kind": "score_calls", "dtype": "f16", "heads": 15,
         "kv_heads": 5, "head_dim": 64, "queries": 4093},
        # The same in f32 at the [9, 2048, 2048] scores of the smaller model.
        {"name": "score_calls_f32", "kind": "score_calls", "dtype": "f32", "heads": 9,
         "kv_heads": 3, "head_dim": 64, "queries": 2048},
        # The normalisations of a large token batch, plain and after the residual add.
        {"name": "norms_f32", "kind": "norms", "dtype": "f32", "tokens": 16384, "hidden": 960},
        # The element-wise and broadcast batch on [4096, 1536], recorded once and replayed.
        {"name": "elementwise_f16", "kind": "elementwise", "dtype": "f16", "tokens": 4096,
         "hidden": 1536, "recorded": True},
        # The front of a prompt: token embedding, head transpose, KV expansion, widening cast.
        {"name": "front_f16", "kind": "front", "dtype": "f16", "layer": 1, "tokens": 2047,
         "vocab": 49152},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["decode_step", "decode", "prefill_layer", "prefill", "prefill", "chunked",
                       "other_head", "score_calls", "norms", "elementwise", "front"])
    dtype = rng.choice(["f16", "f16", "f32"])
    if kind == "decode_step":
        capacity = rng.choice([1024, 2048, 4096])
        return {"kind": kind, "dtype": dtype, "layer": rng.randrange(2),
                "cached": min(_log(rng, 1, capacity), capacity - 1), "capacity": capacity}
    if kind == "prefill_layer":
        return {"kind": kind, "dtype": "f16", "layer": rng.randrange(2),
                "tokens": _log(rng, 16, 4096)}
    if kind == "norms":
        return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 1, 16384),
                "hidden": rng.choice([576, 768, 960])}
    if kind == "elementwise":
        return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 1, 4096),
                "hidden": rng.choice([576, 768, 960, 1535, 1536, 2560]),
                "recorded": rng.random() < 0.5}
    if kind == "front":
        return {"kind": kind, "dtype": dtype, "layer": rng.randrange(2),
                "tokens": _log(rng, 1, 2048), "vocab": 49152}
    heads, kv_heads = rng.choice(HEADS)
    head_dim = rng.choice([64, 64, 128, 96, 32])
    if kind == "score_calls":
        # no more scores than the largest listed call of the type
        most = 15 * 4093 ** 2 if dtype == "f16" else 9 * 2048 ** 2
        queries = _log(rng, 16, int(math.sqrt(most * 64 / (heads * max(64, head_dim)))))
        return {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
                "head_dim": head_dim, "queries": queries}
    batch, cached = 1, 0
    if kind == "decode":
        batch, queries, cached = rng.choice([1, 2, 4, 8]), rng.choice([1, 1, 1, 2, 3]), \
            _log(rng, 16, 4000)
    elif kind == "chunked":
        queries, cached = _log(rng, 16, 512), _log(rng, 256, 3500)
        if heads * head_dim > 32 * 64:
            cached = min(cached, 3000)
    elif kind == "prefill":
        most = 15 * 64 * (4096 if dtype == "f16" else 3001) ** 2
        queries = _log(rng, 16, int(math.sqrt(most / (heads * head_dim))))
    else:
        # a head size off the multiples of 32 up to 128
        head_dim, dtype = rng.choice([48, 80, 80, 112, 256]), "f16"
        queries = _log(rng, 16, int(math.sqrt(8 * 80 * 1021 ** 2 / (heads * head_dim))))
    capacity = -(-(cached + queries) // 64) * 64
    return {"kind": "attention", "dtype": dtype, "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "head_dim": head_dim, "queries": queries, "cached": cached,
            "capacity": capacity}


# ------------------------------------------------------------------ inputs


class _Inputs:
    """Seeded device tensors of one type."""

    def __init__(self, case: dict, seed: int):
        self.dtype = DTYPES[case["dtype"]][0]
        self.rng = torch.Generator(device="cuda")
        self.rng.manual_seed(seed)

    def normal(self, *shape, sigma=1.0):
        x = torch.empty(shape, dtype=self.dtype, device="cuda")
        x.normal_(0.0, sigma, generator=self.rng)
        return x

    def uniform(self, *shape, lo=0.5, hi=1.5):
        x = torch.empty(shape, dtype=self.dtype, device="cuda")
        x.uniform_(lo, hi, generator=self.rng)
        return x

    def scores(self, *shape):
        """Attention logits: N(0, 4), one in a hundred at +20."""
        x = self.normal(*shape, sigma=4.0)
        pick = torch.empty(shape, dtype=torch.float16, device="cuda")
        pick.uniform_(0.0, 1.0, generator=self.rng)
        return x.masked_fill_(pick < 0.01, 20.0)


def _tables(rows: int, head_dim: int):
    inv = THETA ** (-torch.arange(0, head_dim, 2, dtype=torch.float64) / head_dim)
    angle = torch.arange(rows, dtype=torch.float64)[:, None] * inv[None, :]
    return angle.cos().float().cuda(), angle.sin().float().cuda()


def _inputs(case: dict, seed: int) -> dict:
    """The named inputs of a case: device tensors (and host token ids)."""
    r, kind = _Inputs(case, seed), case["kind"]
    if kind in ("decode_step", "prefill_layer"):
        hidden, qh, kvh, ffn = LAYERS[case["layer"]]
        n = 1 if kind == "decode_step" else case["tokens"]
        capacity = case["capacity"] if kind == "decode_step" else n
        cos, sin = _tables(capacity, 64)
        t = {"x": r.normal(n, hidden), "w": r.uniform(hidden), "q": r.normal(n, qh * 64),
             "k": r.normal(n, kvh * 64), "v": r.normal(n, kvh * 64), "cos": cos, "sin": sin,
             "kc": r.normal(1, kvh, capacity, 64), "vc": r.normal(1, kvh, capacity, 64),
             "gate": r.normal(n, ffn), "up": r.normal(n, ffn), "proj": r.normal(n, hidden)}
        if kind == "decode_step":
            t.update(w2=r.uniform(hidden), down=r.normal(n, hidden))
        else:
            t.update(s=r.scores(qh, n, n))
        return t
    if kind == "attention":
        b, d = case["batch"], case["head_dim"]
        kv = (b, case["kv_heads"], case["capacity"], d)
        return {"q": r.normal(b, case["heads"], case["queries"], d), "k": r.normal(*kv),
                "v": r.normal(*kv)}
    if kind == "score_calls":
        n, d = case["queries"], case["head_dim"]
        return {"q": r.normal(1, case["heads"], n, d), "k": r.normal(1, case["kv_heads"], n, d),
                "v": r.normal(1, case["kv_heads"], n, d)}
    if kind == "norms":
        n, h = case["tokens"], case["hidden"]
        return {"x": r.normal(n, h, sigma=2.0), "w": r.uniform(h),
                "r": r.normal(n, h, sigma=2.0)}
    if kind == "elementwise":
        n, h = case["tokens"], case["hidden"]
        return {"a": r.normal(n, h), "b": r.normal(n, h), "bias": r.normal(h)}
    hidden, _, kvh, _ = LAYERS[case["layer"]]
    n = case["tokens"]
    ids = torch.randint(0, case["vocab"], (n,), generator=r.rng, device="cuda")
    return {"table": r.normal(case["vocab"], hidden), "k": r.normal(n, kvh * 64),
            "ids": ids.cpu().numpy().astype(np.uint32)}


def _outputs(case: dict) -> dict:
    """Shapes (and types, where not the case's) of a case's own output buffers."""
    kind = case["kind"]
    if kind in ("decode_step", "prefill_layer"):
        hidden, qh, kvh, ffn = LAYERS[case["layer"]]
        n = 1 if kind == "decode_step" else case["tokens"]
        if kind == "decode_step":
            return {"xn": (n, hidden), "qr": (1, qh, n, 64), "att": (1, qh, n, 64),
                    "sum": (n, hidden), "norm": (n, hidden), "act": (n, ffn),
                    "out": (n, hidden)}
        return {"xn": (n, hidden), "qr": (1, qh, n, 64), "kr": (1, qh, n, 64),
                "vr": (1, qh, n, 64), "p": (qh, n, n), "act": (n, ffn), "out": (n, hidden)}
    if kind == "attention":
        return {"out": (case["batch"], case["heads"], case["queries"], case["head_dim"])}
    if kind == "score_calls":
        h, n = case["heads"], case["queries"]
        return {"s": (1, h, n, n), "p": (1, h, n, n), "out": (1, h, n, case["head_dim"])}
    if kind == "norms":
        n, h = case["tokens"], case["hidden"]
        return {"y": (n, h), "sum": (n, h), "norm": (n, h)}
    if kind == "elementwise":
        n, h = case["tokens"], case["hidden"]
        return {"add": (n, h), "mul": (n, h), "silu": (n, h), "swiglu": (n, h), "biased": (n, h),
                "cast": (n, h)}
    hidden, qh, kvh, _ = LAYERS[case["layer"]]
    n = case["tokens"]
    return {"x": (n, hidden), "k": (1, kvh, n, 64), "kr": (1, qh, n, 64), "cast": (n, hidden)}


def _wrap(tensors: dict) -> dict:
    """The library's view of torch's device memory (an rl_buffer owns nothing)."""
    ctx, out = context(), {}
    names = {torch.float16: np.float16, torch.float32: np.float32}
    for name, t in tensors.items():
        if isinstance(t, torch.Tensor):
            raw = abi.RlBuffer(t.data_ptr(), t.numel(), t.numel() * t.element_size())
            out[name] = abi.DeviceBuffer(ctx, raw, names[t.dtype], tuple(t.shape))
        else:
            out[name] = t
    return out


def prepare(case: dict, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]][0]
    tensors = _inputs(case, seed)
    results = {}
    for name, shape in _outputs(case).items():
        other = torch.float32 if dtype == torch.float16 else torch.float16
        results[name] = torch.empty(shape, dtype=other if name == "cast" else dtype,
                                    device="cuda")
    if case["kind"] in ("decode_step", "prefill_layer"):  # updated in place
        results.update(kc=tensors["kc"], vc=tensors["vc"])
    state = {"case": case, "tensors": tensors, "results": results, "i": _wrap(tensors),
             "o": _wrap(results), "graph": None}
    torch.cuda.synchronize()
    if case.get("recorded"):
        ctx = context()
        ctx.capture_begin()
        _elementwise(ctx, case, state["i"], state["o"])
        state["graph"] = _Graph(ctx)
    return state


class _Graph:
    """A recorded graph, given back with the state that keeps it."""

    def __init__(self, ctx: abi.Context):
        self.ctx, self.handle = ctx, ctx.capture_end()

    def __del__(self):
        if self.ctx.handle:
            self.ctx.graph_destroy(self.handle)


# -------------------------------------------------------------------- runs


def _heads_view(buf, heads: int, n: int):
    """The [1, heads, n, 64] view of [n, heads * 64] projection rows."""
    return buf, (1, heads, n, 64), (n * heads * 64, 64, heads * 64, 1)


def _decode_step(ctx, case, i, o):
    _, qh, kvh, _ = LAYERS[case["layer"]]
    at = case["cached"]
    ctx.rmsnorm(i["x"], i["w"], EPS, o["xn"])
    ctx.qkv_rope_kv_append(_heads_view(i["q"], qh, 1), _heads_view(i["k"], kvh, 1),
                           _heads_view(i["v"], kvh, 1), i["cos"], i["sin"], at, i["kc"], i["vc"],
                           o["qr"])
    ctx.attention(o["qr"], i["kc"], i["vc"], 0.125, at, at + 1, o["att"])
    ctx.add_rmsnorm(i["x"], i["proj"], i["w2"], EPS, o["sum"], o["norm"])
    ctx.swiglu(i["gate"], i["up"], o["act"])
    ctx.add(o["sum"], i["down"], o["out"])


def _prefill_layer(ctx, case, i, o):
    _, qh, kvh, _ = LAYERS[case["layer"]]
    n = case["tokens"]
    ctx.rmsnorm(i["x"], i["w"], EPS, o["xn"])
    ctx.qkv_rope_kv_append_repeat(_heads_view(i["q"], qh, n), _heads_view(i["k"], kvh, n),
                                  _heads_view(i["v"], kvh, n), i["cos"], i["sin"], 0, i["kc"],
                                  i["vc"], qh // kvh, o["qr"], o["kr"], o["vr"])
    ctx.attention_softmax(i["s"], 0.125, 0, o["p"])
    ctx.swiglu(i["gate"], i["up"], o["act"])
    ctx.add(i["x"], i["proj"], o["out"])


def _attention(ctx, case, i, o):
    ctx.attention(i["q"], i["k"], i["v"], 1.0 / math.sqrt(case["head_dim"]), case["cached"],
                  case["cached"] + case["queries"], o["out"])


def _score_calls(ctx, case, i, o):
    ctx.gqa_qk(i["q"], i["k"], None, o["s"])
    ctx.attention_softmax(o["s"], 1.0 / math.sqrt(case["head_dim"]), 0, o["p"])
    ctx.gqa_pv(o["p"], i["v"], o["out"])


def _norms(ctx, case, i, o):
    ctx.rmsnorm(i["x"], i["w"], EPS, o["y"])
    ctx.add_rmsnorm(i["x"], i["r"], i["w"], EPS, o["sum"], o["norm"])


def _elementwise(ctx, case, i, o):
    ctx.add(i["a"], i["b"], o["add"])
    ctx.mul(i["a"], i["b"], o["mul"])
    ctx.silu(i["a"], o["silu"])
    ctx.swiglu(i["a"], i["b"], o["swiglu"])
    ctx.add_broadcast(i["a"], i["bias"], o["biased"])
    ctx.cast(i["a"], o["cast"].dtype, o["cast"])


def _front(ctx, case, i, o):
    _, qh, kvh, _ = LAYERS[case["layer"]]
    n = case["tokens"]
    ctx.embedding(i["table"], i["ids"], o["x"])
    ctx.contiguous(*_heads_view(i["k"], kvh, n), o["k"])
    ctx.repeat_kv(o["k"], qh // kvh, o["kr"])
    ctx.cast(o["x"], o["cast"].dtype, o["cast"])


RUNS = {"decode_step": _decode_step, "prefill_layer": _prefill_layer, "attention": _attention,
        "score_calls": _score_calls, "norms": _norms, "elementwise": _elementwise,
        "front": _front}


def run(state: dict) -> dict:
    if state["graph"] is not None:
        context().graph_launch(state["graph"].handle)
    else:
        case = state["case"]
        RUNS[case["kind"]](context(), case, state["i"], state["o"])
    return state["results"]


# --------------------------------------------------------- work, tolerance


def work(case: dict) -> dict:
    es, kind = DTYPES[case["dtype"]][2], case["kind"]
    flops = 0
    if kind in ("decode_step", "prefill_layer"):
        hidden, qh, kvh, ffn = LAYERS[case["layer"]]
        n = 1 if kind == "decode_step" else case["tokens"]
        tables = 2 * n * 32 * 4
        qkv = 2 * n * (qh + 2 * kvh) * 64  # Q, K, V read once, written once
        if kind == "decode_step":
            keys = case["cached"] + 1
            numel = 9 * n * hidden + qkv + 2 * kvh * case["cached"] * 64 + n * qh * 64 \
                + 3 * n * ffn
            flops = 4 * 64 * qh * keys
        else:
            # the kept half of the scores read, all probabilities written, K and V repeated
            numel = 5 * n * hidden + qkv + 2 * n * qh * 64 + qh * (n * (n + 1) // 2 + n * n) \
                + 3 * n * ffn
        return {"bytes": numel * es + tables, "flops": flops}
    if kind == "attention":
        d, ql, c = case["head_dim"], case["queries"], case["cached"]
        heads = case["batch"] * case["heads"]
        seen = ql * c + ql * (ql + 1) // 2
        numel = 2 * heads * ql * d + 2 * case["batch"] * case["kv_heads"] * (c + ql) * d
        return {"bytes": numel * es, "flops": 4 * d * heads * seen}
    if kind == "score_calls":
        h, n, d = case["heads"], case["queries"], case["head_dim"]
        seen = n * (n + 1) // 2
        numel = 2 * h * n * d + 2 * case["kv_heads"] * n * d + h * (3 * n * n + seen)
        return {"bytes": numel * es, "flops": 4 * d * h * n * n}
    if kind == "norms":
        return {"bytes": 6 * case["tokens"] * case["hidden"] * es, "flops": 0}
    if kind == "elementwise":
        numel = case["tokens"] * case["hidden"]
        return {"bytes": (2 + 5) * numel * es + numel * (6 - es), "flops": 0}
    hidden, qh, kvh, _ = LAYERS[case["layer"]]
    n = case["tokens"]
    return {"bytes": n * (2 * hidden * es + hidden * (6 - es) + (2 * kvh + qh) * 64 * es + 4),
            "flops": 0}


def tolerance(case: dict):
    """Measured against exact() on an MI355X, about four times the error seen:
    f16 results carry their own rounding (and the rounded scores and
    probabilities of the separate calls), f32 results the sums' and e^x's."""
    if case["kind"] == "front":
        return "exact"
    if case["dtype"] == "f16":
        return {"rel": 2e-3} if case["kind"] == "score_calls" else {"rel": 1e-3}
    if case["kind"] == "elementwise":  # its narrowing cast rounds to f16, exactly
        return {"rel": 1e-6}
    return {"rel": 2e-6}


# ------------------------------------------------------------------- exact


def _norm64(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w


def _silu64(x):
    return x / (1.0 + torch.exp(-x))


def _rope64(x, cos, sin):
    """Rotates (even, odd) half pairs of the last dim: [..., n, d] with [n, d / 2] tables."""
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _split64(rows, heads):
    """[n, heads * 64] rows as [1, heads, n, 64] in 64 bits."""
    return rows.double().reshape(rows.shape[0], heads, 64).transpose(0, 1).contiguous()[None]


def _softmax64(s, start):
    """Causal softmax of scaled [n, keys] scores of queries start .. start + n."""
    n, keys = s.shape
    last = torch.arange(start, start + n, device=s.device)[:, None]
    s = s.masked_fill(torch.arange(keys, device=s.device)[None, :] > last, -math.inf)
    return torch.softmax(s, -1)


def _attend64(q, k, v, start, keys):
    """[B, H, n, d] attention over the first `keys` rows, one head at a time."""
    out = torch.empty_like(q)
    group = q.shape[1] // k.shape[1]
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            kt = k[b, h // group, :keys].transpose(0, 1).contiguous()
            s = torch.mm(q[b, h], kt) / math.sqrt(q.shape[-1])
            out[b, h] = torch.mm(_softmax64(s, start), v[b, h // group, :keys].contiguous())
    return out


def exact(case: dict, seed: int) -> dict:
    t, kind = _inputs(case, seed), case["kind"]
    d = {name: x.double() for name, x in t.items()
         if isinstance(x, torch.Tensor) and name not in ("s", "table")}
    if kind in ("decode_step", "prefill_layer"):
        _, qh, kvh, _ = LAYERS[case["layer"]]
        n = d["x"].shape[0]
        at = case.get("cached", 0)
        cos, sin = d["cos"][at:at + n], d["sin"][at:at + n]
        got = {"xn": _norm64(d["x"], d["w"]), "qr": _rope64(_split64(t["q"], qh), cos, sin),
               "act": _silu64(d["gate"]) * d["up"], "kc": d["kc"], "vc": d["vc"]}
        got["kc"][:, :, at:at + n] = _rope64(_split64(t["k"], kvh), cos, sin)
        got["vc"][:, :, at:at + n] = _split64(t["v"], kvh)
        got["sum"] = d["x"] + d["proj"]
        if kind == "decode_step":
            got["att"] = _attend64(got["qr"], got["kc"], got["vc"], at, at + 1)
            got["norm"] = _norm64(got["sum"], d["w2"])
            got["out"] = got["sum"] + d["down"]
            return got
        got["out"] = got.pop("sum")
        got["kr"] = got["kc"].repeat_interleave(qh // kvh, 1)
        got["vr"] = got["vc"].repeat_interleave(qh // kvh, 1)
        got["p"] = torch.empty(t["s"].shape, dtype=torch.float64, device="cuda")
        for h in range(qh):
            got["p"][h] = _softmax64(t["s"][h].double() * 0.125, 0)
        return got
    if kind == "attention":
        return {"out": _attend64(d["q"], d["k"], d["v"], case["cached"],
                                 case["cached"] + case["queries"])}
    if kind == "score_calls":
        h, n, hd = case["heads"], case["queries"], case["head_dim"]
        group = h // case["kv_heads"]
        got = {"s": torch.empty((1, h, n, n), dtype=torch.float64, device="cuda"),
               "p": torch.empty((1, h, n, n), dtype=torch.float64, device="cuda"),
               "out": torch.empty((1, h, n, hd), dtype=torch.float64, device="cuda")}
        for j in range(h):
            kt = d["k"][0, j // group].transpose(0, 1).contiguous()
            got["s"][0, j] = torch.mm(d["q"][0, j], kt)
            got["p"][0, j] = _softmax64(got["s"][0, j] / math.sqrt(hd), 0)
            got["out"][0, j] = torch.mm(got["p"][0, j], d["v"][0, j // group].contiguous())
        return got
    if kind == "norms":
        total = d["x"] + d["r"]
        return {"y": _norm64(d["x"], d["w"]), "sum": total, "norm": _norm64(total, d["w"])}
    if kind == "elementwise":
        silu = _silu64(d["a"])
        return {"add": d["a"] + d["b"], "mul": d["a"] * d["b"], "silu": silu,
                "swiglu": silu * d["b"], "biased": d["a"] + d["bias"], "cast": d["a"]}
    _, qh, kvh, _ = LAYERS[case["layer"]]
    rows = t["table"][torch.from_numpy(t["ids"].astype(np.int64)).cuda()].double()
    k = _split64(t["k"], kvh)
    return {"x": rows, "k": k, "kr": k.repeat_interleave(qh // kvh, 1), "cast": rows}
