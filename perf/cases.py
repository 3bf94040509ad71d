"""The work a user of this library has it do, as cases that can be timed.

Each case names one call (or one block of calls) through the public entry
points of `tiler_amd` on operands already resident on the device, with sizes
from this repository's benchmark, tests and reference cells:

  norm        RMS normalization of bf16 rows, one weight row (Context.rms_norm)
  softmax     f32 softmax over the last axis (Context.softmax_f32)
  embed       bf16 embedding gather (Context.gather)
  linear      bf16 contraction td,od->to, optionally with the fused SiLU
              (Context.contract_bf16)
  attention   one attention block: bf16 scores (contract), widening, the
              scale, f32 softmax, narrowing, bf16 values (contract)
  strict      the f32 contraction under the strict contract, the reference's
              own benchmark cells (Context.contract_strict_f32)
  reduce      the reference's reduction program (x * 1 + 0 into a sum over the
              trailing axis, a flushing and reassociating contract) realized
              and enqueued as a plan, by each of its strategies
  axes        the strict fold of an f32 tensor over chosen axes
              (Context.fold_f32)
  layer       one decoder layer from token ids to logits, in bf16

Device storage is torch's; every launch goes to the bound context's stream.
"""
import math

import torch

from tiler_amd import Context
from tiler_amd import _lib as L
from tiler_amd.realize import prepare_route, realize

EPS_BITS = 0x3727C5AC  # 1e-5 as binary32
EPS = 9.999999747378752e-06

# The layer's widths: the reference's contraction cells (hidden 1024, queries
# 2048, keys and values 1024, MLP 3072, a vocabulary slice of 8192).
HIDDEN, HEADS, KV_HEADS, HEAD_DIM, MLP, VOCAB = 1024, 16, 8, 128, 3072, 8192

_context = None


def context():
    """The program's one bound context."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def listed():
    return [
        # A decode step's normalization: a few rows, all latency.
        {"name": "norm_decode", "kind": "norm", "rows": 16, "extent": 4096},
        # The benchmark's headline: a prefill's hidden states.
        {"name": "norm_prefill", "kind": "norm", "rows": 8192, "extent": 4096},
        # Attention probabilities of 32 heads over 2048 x 2048 scores.
        {"name": "softmax_scores", "kind": "softmax", "rows": 65536, "extent": 2048},
        # Token embedding of a large prefill batch.
        {"name": "embed_prefill", "kind": "embed", "vocab": 128256, "hidden": 4096, "count": 16384},
        # The benchmark's square MLP projection with its activation.
        {"name": "linear_prefill", "kind": "linear", "m": 4096, "n": 4096, "k": 4096, "silu": True},
        # The same projection for a chunk of a prompt: an odd number of tokens.
        {"name": "linear_chunk", "kind": "linear", "m": 300, "n": 4096, "k": 4096, "silu": False},
        # The same projection for one token of each of 48 sequences.
        {"name": "linear_decode", "kind": "linear", "m": 48, "n": 4096, "k": 4096, "silu": False},
        # Grouped-query attention of a 1024-token prompt.
        {"name": "attention_prompt", "kind": "attention", "kv_heads": 8, "group": 2, "queries": 1024,
         "keys": 1024, "dim": 128},
        # The reference's published contraction cell of an MLP input projection.
        {"name": "strict_mlp_in", "kind": "strict", "m": 128, "n": 3072, "k": 1024},
        # The reference's published reduction cell, its workgroup strategy.
        {"name": "reduce_workgroup", "kind": "reduce", "rows": 4096, "extent": 4096, "strategy": "workgroup"},
        # A per-channel sum over every row (a bias gradient, a batch statistic).
        {"name": "axes_channels", "kind": "axes", "outer": 1, "reduced": 4096, "inner": 4096, "variant": "sum"},
        # A whole layer for a short prompt, token ids to logits.
        {"name": "layer_prompt", "kind": "layer", "tokens": 200},
    ]


def _log(rng, lo, hi):
    """A size between lo and hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("norm", "softmax", "embed", "linear", "linear", "attention", "strict", "reduce", "axes",
                       "layer"))
    if kind == "norm":
        extent = rng.choice((512, 1024, 2048, 4096, 8192, _log(rng, 300, 8192)))
        return {"kind": kind, "rows": _log(rng, 1, (1 << 25) // extent), "extent": extent}
    if kind == "softmax":
        extent = rng.choice((512, 1024, 2048, 4096, 131072, _log(rng, 100, 131072)))
        return {"kind": kind, "rows": _log(rng, 1, min(65536, (1 << 26) // extent)), "extent": extent}
    if kind == "embed":
        return {"kind": kind, "vocab": _log(rng, 8192, 128256), "hidden": rng.choice((1024, 2048, 3072, 4096, 1000)),
                "count": _log(rng, 1, 16384)}
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 1, 4096), "n": rng.choice((1024, 2048, 3072, 4096, 8 * _log(rng, 64, 512))),
                "k": rng.choice((1024, 2048, 3072, 4096, 8 * _log(rng, 64, 512))), "silu": rng.random() < 0.5}
    if kind == "attention":
        queries = rng.choice((1, _log(rng, 16, 2048), 64 * _log(rng, 2, 32)))
        keys = max(queries, 8 * _log(rng, 8, 256))
        return {"kind": kind, "kv_heads": rng.choice((4, 8, 16)), "group": rng.choice((1, 2, 4)),
                "queries": queries, "keys": (keys + 7) // 8 * 8, "dim": rng.choice((64, 128))}
    if kind == "strict":
        return {"kind": kind, "m": _log(rng, 1, 512), "n": rng.choice((1024, 2048, 3072, _log(rng, 200, 3072))),
                "k": rng.choice((1024, 2048, 3072, _log(rng, 200, 3072)))}
    if kind == "reduce":
        extent = 16 * _log(rng, 8, 1024)
        return {"kind": kind, "rows": _log(rng, 1, (1 << 24) // extent), "extent": extent,
                "strategy": rng.choice(("serial", "workgroup", "split"))}
    if kind == "axes":
        reduced, inner = _log(rng, 16, 4096), rng.choice((1, _log(rng, 16, 4096), 1024))
        return {"kind": kind, "outer": _log(rng, 1, max(1, (1 << 24) // (reduced * inner))), "reduced": reduced,
                "inner": inner, "variant": rng.choice(("sum", "squared", "maximum"))}
    return {"kind": kind, "tokens": _log(rng, 1, 512)}


# ---------------------------------------------------------------------------
# Inputs

def _normal(g, shape, std=1.0, dtype=torch.bfloat16, mean=0.0):
    """Seeded normal values (made in binary32, a block at a time, then narrowed)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for lo in range(0, flat.numel(), 1 << 26):
        hi = min(flat.numel(), lo + (1 << 26))
        flat[lo:hi] = torch.randn(hi - lo, generator=g, device="cuda").mul_(std).add_(mean)
    return out


def _partitions(extent):
    """The reference's balanced split: the largest divisor at most the root."""
    return max(d for d in range(1, math.isqrt(extent) + 1) if extent % d == 0)


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "norm":
        return {"x": _normal(g, (case["rows"], case["extent"])), "w": _normal(g, (case["extent"],), 0.1, mean=1.0)}
    if kind == "softmax":
        return {"x": _normal(g, (case["rows"], case["extent"]), 3.0, torch.float32)}
    if kind == "embed":
        return {"table": _normal(g, (case["vocab"], case["hidden"]), 0.02),
                "index": torch.randint(0, case["vocab"], (case["count"],), generator=g, device="cuda",
                                       dtype=torch.int32)}
    if kind == "linear":
        return {"a": _normal(g, (case["m"], case["k"])), "b": _normal(g, (case["n"], case["k"]), case["k"] ** -0.5)}
    if kind == "attention":
        h, p, m, n, d = (case[x] for x in ("kv_heads", "group", "queries", "keys", "dim"))
        return {"q": _normal(g, (h, p, m, d)), "k": _normal(g, (h, n, d)), "v": _normal(g, (h, n, d))}
    if kind == "strict":
        return {"a": _normal(g, (case["m"], case["k"]), 1.0, torch.float32),
                "b": _normal(g, (case["n"], case["k"]), 1.0, torch.float32)}
    if kind == "reduce":
        return {"x": _normal(g, (case["rows"], case["extent"]), 1.0, torch.float32)}
    if kind == "axes":
        return {"x": _normal(g, (case["outer"], case["reduced"], case["inner"]), 1.0, torch.float32)}
    t = case["tokens"]
    one = HIDDEN ** -0.5
    return {"ids": torch.randint(0, VOCAB, (t,), generator=g, device="cuda", dtype=torch.int32),
            "table": _normal(g, (VOCAB, HIDDEN)), "norm1": _normal(g, (HIDDEN,), 0.1, mean=1.0),
            "norm2": _normal(g, (HIDDEN,), 0.1, mean=1.0), "norm3": _normal(g, (HIDDEN,), 0.1, mean=1.0),
            "wq": _normal(g, (HEADS * HEAD_DIM, HIDDEN), one), "wk": _normal(g, (KV_HEADS * HEAD_DIM, HIDDEN), one),
            "wv": _normal(g, (KV_HEADS * HEAD_DIM, HIDDEN), one),
            "wo": _normal(g, (HIDDEN, HEADS * HEAD_DIM), (HEADS * HEAD_DIM) ** -0.5),
            "gate": _normal(g, (MLP, HIDDEN), one), "up": _normal(g, (MLP, HIDDEN), one),
            "down": _normal(g, (HIDDEN, MLP), MLP ** -0.5), "head": _normal(g, (VOCAB, HIDDEN), one)}


def _attention_buffers(h, p, m, n, d):
    def new(dtype, *shape):
        return torch.empty(shape, dtype=dtype, device="cuda")
    return {"scores": new(torch.bfloat16, h, p, m, n), "scores32": new(torch.float32, h, p, m, n),
            "scaled": new(torch.float32, h, p, m, n), "probs32": new(torch.float32, h, p, m, n),
            "probs": new(torch.bfloat16, h, p, m, n), "o": new(torch.bfloat16, h, p, m, d),
            "score_form": L.contraction_structure("hpmd", (h, p, m, d), "hnd", (h, n, d), "hpmn"),
            "value_form": L.contraction_structure("hpmn", (h, p, m, n), "hnd", (h, n, d), "hpmd")}


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]

    def new(dtype, *shape):
        return torch.empty(shape, dtype=dtype, device="cuda")

    if kind == "norm":
        s["y"] = new(torch.bfloat16, case["rows"], case["extent"])
    elif kind == "softmax":
        s["y"] = new(torch.float32, case["rows"], case["extent"])
    elif kind == "embed":
        s["y"] = new(torch.bfloat16, case["count"], case["hidden"])
    elif kind == "linear":
        s["c"] = new(torch.bfloat16, case["m"], case["n"])
    elif kind == "attention":
        s.update(_attention_buffers(*(case[x] for x in ("kv_heads", "group", "queries", "keys", "dim"))))
    elif kind == "strict":
        s["c"] = new(torch.float32, case["m"], case["n"])
    elif kind == "reduce":
        s["y"] = new(torch.float32, case["rows"])
        p = _partitions(case["extent"])
        c = case["extent"] // p
        shape = {"serial": {"topology": L.SUM_SERIAL, "grouping": (2,)},
                 "workgroup": {"topology": L.SUM_COOPERATIVE, "grouping": (2, p, c)},
                 "split": {"topology": L.SUM_MULTIPASS, "grouping": (2, p, c)}}[case["strategy"]]
        rz = realize(L.PROGRAM_FOLD, (case["rows"], case["extent"]), ctx=context(), variant=L.FOLD_FMA, rank=2,
                     scalars=(0x3F800000, 0), flags=L.REGION_ALIGNED16, permissions=L.PERMITS_REASSOCIATION,
                     input_subnormals=L.SUBNORMALS_FLUSH_SIGN, result_subnormals=L.SUBNORMALS_FLUSH_SIGN, **shape)
        s["plan"] = _Plan(prepare_route(context(), rz, [s["x"].data_ptr(), s["y"].data_ptr()]
                                        + [None] * (len(rz.slots) - 2)))
    elif kind == "axes":
        s["y"] = new(torch.float32, case["outer"], case["inner"])
    else:
        t, bf16 = case["tokens"], torch.bfloat16
        s.update(_attention_buffers(KV_HEADS, HEADS // KV_HEADS, t, t, HEAD_DIM))
        for name, width in (("x", HIDDEN), ("h", HIDDEN), ("x1", HIDDEN), ("h1", HIDDEN), ("x2", HIDDEN),
                            ("h2", HIDDEN), ("od", HIDDEN), ("down_out", HIDDEN), ("q_rows", HEADS * HEAD_DIM),
                            ("k_rows", KV_HEADS * HEAD_DIM), ("v_rows", KV_HEADS * HEAD_DIM),
                            ("o_rows", HEADS * HEAD_DIM), ("gate_out", MLP), ("up_out", MLP), ("mid", MLP),
                            ("logits", VOCAB)):
            s[name] = new(bf16, t, width)
        s["q"] = new(bf16, HEADS, t, HEAD_DIM)
        s["k"] = new(bf16, KV_HEADS, t, HEAD_DIM)
        s["v"] = new(bf16, KV_HEADS, t, HEAD_DIM)
    s["case"] = case
    return s


class _Plan:
    """A routed plan that gives its scratch back with the state."""

    def __init__(self, plan):
        self.plan = plan

    def __del__(self):
        try:
            self.plan.release()
        except Exception:
            pass


# ---------------------------------------------------------------------------
# One pass

def _attend(ctx, s, h, p, m, n, d, q, k, v, o):
    total = h * p * m * n
    ctx.contract(L.BF16, s["score_form"], q, k, s["scores"].data_ptr(), permissions=L.PERMITS_REASSOCIATION)
    ctx.convert(L.CONVERT_WIDEN_BF16_F32, s["scores"].data_ptr(), total, s["scores32"].data_ptr())
    ctx.map(L.MAP_SCALE_BIAS, L.F32, s["scores32"].data_ptr(), total, s["scaled"].data_ptr(), a=d ** -0.5, b=0.0)
    ctx.softmax_f32(s["scaled"].data_ptr(), h * p * m, n, s["probs32"].data_ptr())
    ctx.convert(L.CONVERT_NARROW_F32_BF16, s["probs32"].data_ptr(), total, s["probs"].data_ptr())
    ctx.contract(L.BF16, s["value_form"], s["probs"].data_ptr(), v, o, permissions=L.PERMITS_REASSOCIATION)


def _run_layer(ctx, s, t):
    at = {name: v.data_ptr() for name, v in s.items() if isinstance(v, torch.Tensor)}
    bf16 = L.BF16

    def linear(x, w, out, n, k, epilogue=L.EPILOGUE_NONE):
        ctx.contract_bf16(at[x], at[w], t, n, k, at[out], epilogue)

    def heads(src, dst, count):  # [t, count, dim] -> [count, t, dim]
        ctx.reindex(at[src], t * count * HEAD_DIM, (count, t, HEAD_DIM), (HEAD_DIM, count * HEAD_DIM, 1), 0, 2, at[dst])

    ctx.gather(at["table"], 1, VOCAB, HIDDEN, 2, at["ids"], t, at["x"], index_signed=True)
    ctx.rms_norm(bf16, at["x"], at["norm1"], t, HIDDEN, EPS_BITS, at["h"])
    linear("h", "wq", "q_rows", HEADS * HEAD_DIM, HIDDEN)
    linear("h", "wk", "k_rows", KV_HEADS * HEAD_DIM, HIDDEN)
    linear("h", "wv", "v_rows", KV_HEADS * HEAD_DIM, HIDDEN)
    heads("q_rows", "q", HEADS)
    heads("k_rows", "k", KV_HEADS)
    heads("v_rows", "v", KV_HEADS)
    _attend(ctx, s, KV_HEADS, HEADS // KV_HEADS, t, t, HEAD_DIM, at["q"], at["k"], at["v"], at["o"])
    ctx.reindex(at["o"], t * HEADS * HEAD_DIM, (t, HEADS, HEAD_DIM), (HEAD_DIM, t * HEAD_DIM, 1), 0, 2, at["o_rows"])
    linear("o_rows", "wo", "od", HIDDEN, HEADS * HEAD_DIM)
    ctx.map(L.MAP_ADD, bf16, at["x"], t * HIDDEN, at["x1"], x2=at["od"])
    ctx.rms_norm(bf16, at["x1"], at["norm2"], t, HIDDEN, EPS_BITS, at["h1"])
    linear("h1", "gate", "gate_out", MLP, HIDDEN, L.EPILOGUE_SILU)
    linear("h1", "up", "up_out", MLP, HIDDEN)
    ctx.map(L.MAP_MULTIPLY, bf16, at["gate_out"], t * MLP, at["mid"], x2=at["up_out"])
    linear("mid", "down", "down_out", HIDDEN, MLP)
    ctx.map(L.MAP_ADD, bf16, at["x1"], t * HIDDEN, at["x2"], x2=at["down_out"])
    ctx.rms_norm(bf16, at["x2"], at["norm3"], t, HIDDEN, EPS_BITS, at["h2"])
    linear("h2", "head", "logits", VOCAB, HIDDEN)
    return {"hidden": s["x2"], "logits": s["logits"]}


def run(s):
    case, ctx = s["case"], context()
    kind = case["kind"]
    if kind == "norm":
        ctx.rms_norm(L.BF16, s["x"].data_ptr(), s["w"].data_ptr(), case["rows"], case["extent"], EPS_BITS,
                     s["y"].data_ptr(), weight_broadcast=True)
        return s["y"]
    if kind == "softmax":
        ctx.softmax_f32(s["x"].data_ptr(), case["rows"], case["extent"], s["y"].data_ptr())
        return s["y"]
    if kind == "embed":
        ctx.gather(s["table"].data_ptr(), 1, case["vocab"], case["hidden"], 2, s["index"].data_ptr(), case["count"],
                   s["y"].data_ptr(), index_signed=True)
        return s["y"]
    if kind == "linear":
        ctx.contract_bf16(s["a"].data_ptr(), s["b"].data_ptr(), case["m"], case["n"], case["k"], s["c"].data_ptr(),
                          L.EPILOGUE_SILU if case["silu"] else L.EPILOGUE_NONE)
        return s["c"]
    if kind == "attention":
        _attend(ctx, s, *(case[x] for x in ("kv_heads", "group", "queries", "keys", "dim")), s["q"].data_ptr(),
                s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr())
        return s["o"]
    if kind == "strict":
        ctx.contract_strict_f32(s["a"].data_ptr(), s["b"].data_ptr(), case["m"], case["n"], case["k"],
                                s["c"].data_ptr())
        return s["c"]
    if kind == "reduce":
        s["plan"].plan.enqueue()
        return s["y"]
    if kind == "axes":
        variant = {"sum": L.FOLD_SUM, "squared": L.FOLD_SQUARED, "maximum": L.FOLD_MAXIMUM}[case["variant"]]
        ctx.fold_f32(variant, s["x"].data_ptr(), (case["outer"], case["reduced"], case["inner"]), (1,),
                     s["y"].data_ptr())
        return s["y"]
    return _run_layer(ctx, s, case["tokens"])


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what its outputs may be off by

def work(case):
    kind = case["kind"]
    if kind == "norm":
        n = case["rows"] * case["extent"]
        return {"bytes": 4 * n + 2 * case["extent"], "flops": 4 * n}
    if kind == "softmax":
        n = case["rows"] * case["extent"]
        return {"bytes": 8 * n, "flops": 5 * n}
    if kind == "embed":
        return {"bytes": case["count"] * (4 * case["hidden"] + 4), "flops": 0}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "attention":
        h, p, m, n, d = (case[x] for x in ("kv_heads", "group", "queries", "keys", "dim"))
        return {"bytes": 2 * h * (2 * p * m * d + 2 * n * d), "flops": 4 * h * p * m * n * d}
    if kind == "strict":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "reduce":
        return {"bytes": 4 * case["rows"] * (case["extent"] + 1), "flops": 3 * case["rows"] * case["extent"]}
    if kind == "axes":
        n = case["outer"] * case["reduced"] * case["inner"]
        return {"bytes": 4 * n + 4 * case["outer"] * case["inner"], "flops": n}
    t, qd, kvd = case["tokens"], HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    weights = HIDDEN * (2 * qd + 2 * kvd + 3 * MLP + VOCAB)
    return {"bytes": 2 * weights + 2 * t * (2 * HIDDEN + VOCAB) + 4 * t,
            "flops": 2 * t * weights + 4 * HEADS * t * t * HEAD_DIM}


def tolerance(case):
    kind = case["kind"]
    if kind in ("embed", "strict", "reduce", "axes"):
        # bytes moved, or a fold whose order and grouping the contract fixes
        return "exact"
    if kind == "softmax":
        # binary32 sums in another order
        return {"rel": 2e-6, "max": 1e-5}
    if kind in ("norm", "linear"):
        # one bf16 rounding of a binary32 value: another summation order moves
        # a value across a rounding boundary here and there, by one bf16 step
        return {"rel": 1e-3, "max": 0.01}
    if kind == "attention":
        # three bf16 roundings (scores, probabilities, result)
        return {"rel": 2e-3, "max": 0.05}
    # a layer: some twenty bf16 roundings, each carried through what follows
    return {"rel": 1e-2, "max": 0.2}


def exact(case, seed):
    """The same results in 64 bits by plain torch."""
    kind = case["kind"]
    if kind == "embed":
        return None
    s = _inputs(case, seed)
    x = {name: v.double() for name, v in s.items() if v.is_floating_point()}

    def norm(v, w):
        return v * torch.rsqrt((v * v).mean(-1, keepdim=True) + EPS) * w

    if kind == "norm":
        return norm(x["x"], x["w"])
    if kind == "softmax":
        return torch.softmax(x["x"], -1)
    if kind == "linear":
        c = x["a"] @ x["b"].T
        return torch.nn.functional.silu(c) if case["silu"] else c
    if kind == "strict":
        return x["a"] @ x["b"].T
    if kind == "reduce":
        return x["x"].sum(-1)
    if kind == "axes":
        v = x["x"]
        return v.amax(1) if case["variant"] == "maximum" else (v * v if case["variant"] == "squared" else v).sum(1)

    def attend(q, k, v):  # q [h, p, m, d], k and v [h, n, d]
        out = torch.empty_like(q)
        for i in range(q.shape[0]):
            for j in range(q.shape[1]):
                out[i, j] = torch.softmax(q[i, j] @ k[i].T * q.shape[-1] ** -0.5, -1) @ v[i]
        return out

    if kind == "attention":
        return attend(x["q"], x["k"], x["v"])
    t, group = case["tokens"], HEADS // KV_HEADS
    hidden = x["table"][s["ids"].long()]
    h = norm(hidden, x["norm1"])
    q = (h @ x["wq"].T).view(t, KV_HEADS, group, HEAD_DIM).permute(1, 2, 0, 3).contiguous()
    k = (h @ x["wk"].T).view(t, KV_HEADS, HEAD_DIM).permute(1, 0, 2).contiguous()
    v = (h @ x["wv"].T).view(t, KV_HEADS, HEAD_DIM).permute(1, 0, 2).contiguous()
    o = attend(q, k, v).permute(2, 0, 1, 3).reshape(t, HEADS * HEAD_DIM)
    hidden = hidden + o @ x["wo"].T
    h = norm(hidden, x["norm2"])
    mid = torch.nn.functional.silu(h @ x["gate"].T) * (h @ x["up"].T)
    hidden = hidden + mid @ x["down"].T
    return {"hidden": hidden, "logits": norm(hidden, x["norm3"]) @ x["head"].T}
