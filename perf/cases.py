"""Timed cases of the column reduction, through the package's public functions.

A case is one call (or the two calls of a pruning step) as a serving or evaluation program makes it:
`flash_colreduce`, `flash_colreduce_multi`, `topk_keep_mask`.  `listed()` spans the shapes of the named
workloads, the benchmark table and the tests, from calls that are all launch latency to ones that fill the
chip for milliseconds; `draw()` gives more of the same ranges.
"""
from __future__ import annotations

import math

import torch

from flash_colreduce_amd import flash_colreduce, flash_colreduce_multi
from flash_colreduce_amd.flash import topk_keep_mask

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_BYTES = {"float16": 2, "bfloat16": 2, "float32": 4}

# What a drawn case may cost at most (the largest listed one): work on the matrix units in 16-bit
# equivalents, and bytes.
_MOST_FLOPS = 4.4e12
_MOST_BYTES = 2.2e9


def _case(name, call, b, h, m, n, d, dtype, reduction, causal, keys="normal", layout="bhsd", keep=0.0):
    c = dict(call=call, B=b, H=h, M=m, N=n, D=d, dtype=dtype, reduction=reduction, causal=causal, keys=keys,
             layout=layout, keep=keep)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call of the named workloads: fp32, two heads, one short sequence.  Launches and latency.
        _case("tiny fp32", "reduce", 1, 2, 256, 256, 64, "float32", "sum", False),
        # A batch of short sequences without a mask, as an encoder gives them; the mean over the queries.
        _case("short batch fp16", "reduce", 8, 16, 512, 512, 64, "float16", "mean", False),
        # The last 128 queries of a prompt against its cache: which keys did the observation window look at.
        _case("window 128x4096 fp16", "reduce", 1, 32, 128, 4096, 128, "float16", "mean", True),
        # The same with 64 queries over a serving batch of long caches: reading the keys is the work.
        _case("window batch 64x16384 fp16", "reduce", 16, 32, 64, 16384, 128, "float16", "sum", True),
        # One decoded token per sequence, ragged cache length: the accumulated-attention score of every key.
        _case("token 1x9001 bf16", "reduce", 8, 32, 1, 9001, 128, "bfloat16", "sum", True),
        # A prefill chunk of 512 queries against the cache so far.
        _case("chunk 512x32768 bf16", "reduce", 1, 32, 512, 32768, 128, "bfloat16", "sum", True),
        # Prefill of one prompt: the headline workload.
        _case("prefill 8192 fp16", "reduce", 1, 32, 8192, 8192, 128, "float16", "sum", True),
        # The largest: long-context cache pruning, mean and maximum of the same attention matrix.
        _case("long 32768 bf16", "multi", 1, 32, 32768, 32768, 128, "bfloat16", "mean,max", True, keys="offset"),
        # Visual-token pruning of a small batch: ragged length, projections viewed as heads (token-major
        # memory), heavy-hitter keys, then the mask of the quarter of the keys to keep.
        _case("prune 2929 bf16", "prune", 2, 24, 2929, 2929, 128, "bfloat16", "mean", True, keys="sinks",
              layout="bshd", keep=0.25),
        # Full-precision operands, the benchmark table's first shape.
        _case("fp32 1024", "reduce", 1, 32, 1024, 1024, 128, "float32", "sum", False),
        # Wide heads.
        _case("wide heads 2048x256 bf16", "reduce", 2, 16, 2048, 2048, 256, "bfloat16", "sum", True),
        # Only the selection: the keep-mask of a quarter of 32768 columns from 32 heads' scores.
        _case("keep 32x32768 fp16", "keep", 1, 32, 1, 32768, 8, "float16", "", False, keep=0.25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A length in [lo, hi]: any number, or a multiple of 64, half of the time each."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < 0.5 else min(hi, max(lo, (v + 63) // 64 * 64))


def draw(rng):
    kind = rng.choice(["short", "window", "token", "chunk", "prefill", "prefill", "prune", "keep"])
    dtype = rng.choice(["float16", "float16", "float16", "bfloat16", "bfloat16", "bfloat16", "float32"])
    d = rng.choice([64, 64, 80, 96, 128, 128, 128, 128, 192, 256])
    h = rng.choice([8, 12, 16, 24, 32, 32, 40])
    b = _log_int(rng, 1, 16)
    reduction = rng.choice(["sum", "sum", "mean", "mean", "max", "mean,max"])
    layout = rng.choice(["bhsd", "bshd"])
    keys = rng.choice(["normal", "sinks", "offset"])
    causal, keep, call = True, 0.0, "multi" if "," in reduction else "reduce"
    if kind == "keep":
        return _case("", "keep", b, h, 1, _length(rng, 512, 131072), 8, dtype, "", False,
                     keep=rng.choice([0.1, 0.25, 0.5]))
    if kind == "short":
        h = rng.choice([2, 8, 16, 32])
        m = n = _length(rng, 64, 1024)
        causal = rng.random() < 0.3
    elif kind == "window":
        m, n = _length(rng, 16, 128), _length(rng, 1024, 65536)
    elif kind == "token":
        m, n = 1, _length(rng, 1024, 65536)
    elif kind == "chunk":
        m, n = _length(rng, 129, 1024), _length(rng, 2048, 65536)
    else:
        m = n = _length(rng, 1024, 16384)
        causal = rng.random() < 0.75
        if kind == "prune":
            call, reduction, keep = "prune", reduction.split(",")[0], rng.choice([0.1, 0.25, 0.5])
    c = _case("", call, b, h, m, n, d, dtype, reduction, causal, keys, layout, keep)
    while True:
        w = work(c)
        if w["flops"] * (16 if dtype == "float32" else 1) <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return c
        if c["B"] > 1:
            c["B"] //= 2
        elif c["H"] > 8:
            c["H"] = 8
        else:
            c["N"] = max(c["N"] // 2, 1024)
            c["M"] = min(c["M"], c["N"])


def _heads(c, rows, g):
    """(B, H, rows, D) of N(0,1) draws; 'bshd' is token-major memory seen as heads."""
    shape = (c["B"], c["H"], rows, c["D"]) if c["layout"] == "bhsd" else (c["B"], rows, c["H"], c["D"])
    x = torch.randn(shape, generator=g, device="cuda", dtype=_DTYPES[c["dtype"]])
    return x if c["layout"] == "bhsd" else x.transpose(1, 2)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    c = dict(case)
    state = {"case": c, "kept": max(1, int(c["keep"] * c["N"]))}
    if c["call"] == "keep":
        # column scores as the reduction leaves them: positive, skewed, in the operands' type
        x = torch.randn((c["B"], c["H"], c["N"]), generator=g, device="cuda").exp()
        state["scores"] = x.to(_DTYPES[c["dtype"]])
        return state
    state["q"], k = _heads(c, c["M"], g), _heads(c, c["N"], g)
    if c["keys"] == "sinks":     # one key in a hundred draws four times the attention logits, the first one eight times
        idx = torch.randint(0, c["N"], (max(1, c["N"] // 100),), generator=g, device="cuda").unique()
        k[:, :, idx] *= 4
        k[:, :, 0] *= 2
    elif c["keys"] == "offset":  # every key of a head shares an offset
        k += 0.5 * torch.randn((c["B"], c["H"], 1, c["D"]), generator=g, device="cuda", dtype=k.dtype)
    state["k"] = k
    return state


def run(state):
    c = state["case"]
    if c["call"] == "keep":
        mask, threshold = topk_keep_mask(state["scores"], state["kept"], return_threshold=True)
        return mask, threshold
    if c["call"] == "multi":
        return flash_colreduce_multi(state["q"], state["k"], c["reduction"].split(","), is_causal=c["causal"])
    scores = flash_colreduce(state["q"], state["k"], c["reduction"], is_causal=c["causal"])
    if c["call"] == "prune":
        return scores, topk_keep_mask(scores, state["kept"])
    return scores


def work(case):
    """One product per visible score and every operand and result once.  (A call whose scores do not fit the
    chip forms them twice, once for the row statistics and once for the columns; that is not counted.)"""
    c = case
    bh, m, n, d, e = c["B"] * c["H"], c["M"], c["N"], c["D"], _BYTES[c["dtype"]]
    if c["call"] == "keep":
        return {"bytes": bh * (n * (e + 1) + 4), "flops": 0}
    seen = m * n
    if c["causal"]:
        off = max(n - m, 0)
        seen = sum(min(n, i + off + 1) for i in range(m))
    results = (2 if c["call"] == "multi" else 1) * bh * n * e + (bh * n if c["call"] == "prune" else 0)
    return {"bytes": bh * (m + n) * d * e + results, "flops": 2 * bh * seen * d}


def tolerance(case):
    """Scores are rounded to the operands' type, so a last-bit difference of the fp32 sums moves a value by
    one unit there (two where a mean divides the rounded sum): 2^-11 of the value for fp16, 2^-8 for bf16."""
    if case["call"] == "keep":
        return "exact"
    t = {"float16": {"rel": 1e-3, "max": 4e-3}, "bfloat16": {"rel": 8e-3, "max": 2e-2},
         "float32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]
    if case["call"] == "prune":
        t = dict(t, differ=5e-3)   # columns at the threshold change sides with their last bit
    return t
