"""The calls whose time counts for a user of this library: GEMM, fused back-to-back GEMM,
flash-attention forward, split-KV decoding and scatter_nd, each through tilefusion_amd.ops as a
program calls it, from the smallest problem of the documentation to the largest benchmark.

A case is a dict of plain values; `op` says which function it calls and the other keys are its sizes,
types and options.  `listed()` names twelve of them, `draw()` gives further ones of the same ranges.
"""

import math

import torch

from tilefusion_amd import ops

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# Bounds of a drawn case, so that none costs more than the largest listed ones.
MAX_GEMM_FLOPS = 2.0 * 4096 ** 3
MAX_FUSED_FLOPS = 4.0 * 8192 * 8192 * 128
MAX_ATTENTION_FLOPS = 4.0 * 64 * 4096 * 4096 * 128
MAX_DECODE_BYTES = 4.0 * 512 * 32768 * 128


def listed():
    return [
        # The documentation's first example, one output tile: the smallest call, all latency.
        {"name": "gemm_readme_tile", "op": "gemm", "m": 128, "n": 64, "k": 256, "dtype": "fp16", "out": "fp32"},
        # A linear layer over the rows of one decoding step: few rows, every weight read once.
        {"name": "gemm_few_rows", "op": "gemm", "m": 32, "n": 4096, "k": 4096, "dtype": "bf16", "out": "bf16"},
        # A layer over packed tokens: a row count of no particular divisor, widths that are multiples
        # of 8 but not of a tile, and the fp32 result that the op has by default.
        {"name": "gemm_ragged", "op": "gemm", "m": 2999, "n": 1544, "k": 1032, "dtype": "fp16", "out": "fp32"},
        # The repository's GEMM benchmark.
        {"name": "gemm_4096", "op": "gemm", "m": 4096, "n": 4096, "k": 4096, "dtype": "fp16", "out": "fp16"},
        # The repository's fused benchmark: a long batch of rows through two small layers.
        {"name": "fused_16384_rows", "op": "fused", "batch": 1, "m": 16384, "n": 128, "k": 128, "p": 128, "dtype": "fp16"},
        # The wide-intermediate end of the fused sweep, with a row count that no tile divides.
        {"name": "fused_wide_ragged", "op": "fused", "batch": 1, "m": 4000, "n": 4096, "k": 128, "p": 128, "dtype": "bf16"},
        # The repository's attention benchmark, its key stored [D, Lkv] as the op takes it.
        {"name": "attention_4096", "op": "attention", "bh": 64, "lq": 4096, "lkv": 4096, "d": 128, "dtype": "fp16",
         "causal": False, "key": "transposed"},
        # Causal prefill of an odd prompt length; the key is a transposed view of a [Lkv, D] tensor.
        {"name": "attention_causal_odd", "op": "attention", "bh": 64, "lq": 1337, "lkv": 1337, "d": 64, "dtype": "bf16",
         "causal": True, "key": "view"},
        # A wide head.
        {"name": "attention_wide_head", "op": "attention", "bh": 32, "lq": 1024, "lkv": 1024, "d": 256, "dtype": "bf16",
         "causal": True, "key": "view"},
        # The repository's decoding benchmark: 8 GiB of keys and values, the largest call.
        {"name": "decode_32768", "op": "decode", "bh": 512, "lkv": 32768, "d": 128, "splits": 64, "dtype": "fp16"},
        # Decoding near the start of a conversation with the default split count.
        {"name": "decode_short", "op": "decode", "bh": 32, "lkv": 1999, "d": 64, "splits": 64, "dtype": "bf16"},
        # Accumulating rows into a table at indices that repeat as word frequencies do: the gradient
        # of an embedding.
        {"name": "scatter_embedding", "op": "scatter", "rows": 32000, "width": 1024, "updates": 8192, "dtype": "bf16"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(x, of):
    return max(of, x // of * of)


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "fused", "attention", "attention", "decode", "scatter"])
    return {"gemm": _draw_gemm, "fused": _draw_fused, "attention": _draw_attention, "decode": _draw_decode,
            "scatter": _draw_scatter}[op](rng)


def _draw_gemm(rng):
    # any row count; layer widths are mostly multiples of 64, otherwise of 8 (n: now and then odd)
    while True:
        m, n, k = _log_int(rng, 1, 8192), _log_int(rng, 64, 8192), _log_int(rng, 64, 8192)
        if rng.random() < 0.4:
            m = _multiple(m, 64)
        if rng.random() < 0.6:
            n, k = _multiple(n, 64), _multiple(k, 64)
        else:
            n, k = (n if rng.random() < 0.3 else _multiple(n, 8)), _multiple(k, 8)
        if 2.0 * m * n * k <= MAX_GEMM_FLOPS:
            break
    dtype = rng.choice(["fp16", "bf16"])
    return {"op": "gemm", "m": m, "n": n, "k": k, "dtype": dtype, "out": rng.choice(["fp32", dtype])}


def _draw_fused(rng):
    # K and P are the narrow dimensions of the fused form; N runs over the sweep's range
    while True:
        batch = rng.choice([1, 1, 1, 2, 8])
        m, n = _log_int(rng, 64, 32768), _multiple(_log_int(rng, 64, 8192), 16)
        if rng.random() < 0.6:
            m, n = _multiple(m, 64), _multiple(n, 64)
        k, p = rng.choice([(128, 128), (128, 128), (64, 64), (64, 128), (96, 48), (48, 80)])
        if 2.0 * batch * m * n * (k + p) <= MAX_FUSED_FLOPS:
            break
    return {"op": "fused", "batch": batch, "m": m, "n": n, "k": k, "p": p, "dtype": rng.choice(["fp16", "bf16"])}


def _draw_attention(rng):
    d = rng.choice([64, 64, 80, 96, 128, 128, 128, 160, 256])
    most = MAX_ATTENTION_FLOPS if d <= 128 else MAX_ATTENTION_FLOPS / 8
    while True:
        bh, lkv = _log_int(rng, 8, 128), _log_int(rng, 128, 8192)
        causal = rng.random() < 0.5
        # self-attention, or a shorter block of queries against a longer key range
        lq = lkv if causal or rng.random() < 0.6 else _log_int(rng, 16, lkv)
        if d > 128:
            lq, lkv = _multiple(lq, 32), _multiple(lkv, 32)   # what the op takes above 128
        elif rng.random() < 0.6:
            lq, lkv = _multiple(lq, 64), _multiple(lkv, 64)
        if causal:
            lq = lkv
        if 4.0 * bh * lq * lkv * d <= most:
            break
    return {"op": "attention", "bh": bh, "lq": lq, "lkv": lkv, "d": d, "dtype": rng.choice(["fp16", "bf16"]),
            "causal": causal, "key": rng.choice(["transposed", "view"])}


def _draw_decode(rng):
    while True:
        bh, lkv, d = _log_int(rng, 8, 1024), _log_int(rng, 128, 65536), rng.choice([128, 128, 64])
        if 4.0 * bh * lkv * d <= MAX_DECODE_BYTES:
            break
    return {"op": "decode", "bh": bh, "lkv": lkv, "d": d, "splits": rng.choice([64, 64, 16, 8]),
            "dtype": rng.choice(["fp16", "bf16"])}


def _draw_scatter(rng):
    while True:
        rows, width, updates = _log_int(rng, 64, 131072), _log_int(rng, 16, 4096), _log_int(rng, 64, 65536)
        if rows * width <= 1 << 28 and updates * width <= 1 << 26:
            break
    return {"op": "scatter", "rows": rows, "width": width, "updates": updates,
            "dtype": rng.choice(["fp32", "fp16", "bf16"])}


def _randn(g, *shape, dtype, scale=1.0):
    x = torch.randn(*shape, device=DEVICE, dtype=dtype, generator=g)
    return x if scale == 1.0 else x.mul_(scale)


def _tile(extent, most=64):
    """A tile size as a caller of the reference's signatures picks it: a power of two that divides."""
    t = 1
    while t < most and extent % (2 * t) == 0:
        t *= 2
    return t


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    op = case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"op": op, "a": _randn(g, m, k, dtype=dtype, scale=k ** -0.5), "b": _randn(g, n, k, dtype=dtype),
                "c": torch.empty(m, n, device=DEVICE, dtype=DTYPES[case["out"]]),
                "tiles": (_tile(m), _tile(n), _tile(k))}
    if op == "fused":
        batch, m, n, k, p = (case[x] for x in ("batch", "m", "n", "k", "p"))
        lead = (batch,) if batch > 1 else ()
        return {"op": op, "a": _randn(g, *lead, m, k, dtype=dtype, scale=k ** -0.5), "b": _randn(g, *lead, n, k, dtype=dtype),
                "c": _randn(g, *lead, p, n, dtype=dtype, scale=n ** -0.5),
                "d": torch.empty(*lead, m, p, device=DEVICE, dtype=dtype),
                "tiles": (_tile(m), _tile(n), _tile(k), _tile(p))}
    if op == "attention":
        bh, lq, lkv, d = (case[x] for x in ("bh", "lq", "lkv", "d"))
        q, v = _randn(g, bh, lq, d, dtype=dtype), _randn(g, bh, lkv, d, dtype=dtype)
        if case["key"] == "transposed":
            key = _randn(g, bh, d, lkv, dtype=dtype)
        else:
            key = _randn(g, bh, lkv, d, dtype=dtype).transpose(-1, -2)
        return {"op": op, "q": q, "k": key, "v": v,
                "options": (_tile(lq), _tile(lkv), d, d, 1.0 / math.sqrt(d), case["causal"])}
    if op == "decode":
        bh, lkv, d = case["bh"], case["lkv"], case["d"]
        return {"op": op, "q": _randn(g, bh, 1, d, dtype=dtype), "k": _randn(g, bh, lkv, d, dtype=dtype),
                "v": _randn(g, bh, lkv, d, dtype=dtype), "splits": case["splits"]}
    rows, width, updates = case["rows"], case["width"], case["updates"]
    # log-uniform row numbers: row i is hit about as often as the i-th most frequent word
    u = torch.rand(updates, device=DEVICE, dtype=torch.float64, generator=g)
    index = (torch.pow(float(rows), u).long() - 1).clamp_(0, rows - 1)
    return {"op": op, "data": _randn(g, rows, width, dtype=dtype), "index": index.unsqueeze(1),
            "updates": _randn(g, updates, width, dtype=dtype, scale=1.0 / 64)}


def run(state):
    op = state["op"]
    if op == "gemm":
        ops.gemm(state["a"], state["b"], state["c"], *state["tiles"], 2, 1)
        return state["c"]
    if op == "fused":
        ops.fused_two_gemms(state["a"], state["b"], state["c"], state["d"], *state["tiles"])
        return state["d"]
    if op == "attention":
        return ops.flash_attention(state["q"], state["k"], state["v"], *state["options"])
    if op == "decode":
        return ops.flash_decode(state["q"], state["k"], state["v"], state["splits"])
    ops.scatter_nd(state["data"], state["index"], state["updates"])
    return state["data"]


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    op = case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + n * k) * size + m * n * (4 if case["out"] == "fp32" else 2), "flops": 2.0 * m * n * k}
    if op == "fused":
        batch, m, n, k, p = (case[x] for x in ("batch", "m", "n", "k", "p"))
        return {"bytes": batch * (m * k + n * k + n * p + m * p) * size, "flops": 2.0 * batch * m * n * (k + p)}
    if op == "attention":
        bh, lq, lkv, d = (case[x] for x in ("bh", "lq", "lkv", "d"))
        pairs = lq * (lq + 1) / 2 if case["causal"] else lq * lkv
        return {"bytes": bh * (2 * lq + 2 * lkv) * d * size, "flops": 4.0 * bh * pairs * d}
    if op == "decode":
        bh, lkv, d = case["bh"], case["lkv"], case["d"]
        return {"bytes": bh * (2 * lkv + 2) * d * size, "flops": 4.0 * bh * lkv * d}
    rows, width, updates = case["rows"], case["width"], case["updates"]
    # of `updates` log-uniform draws this many rows are hit at least once, on average
    hit = sum(1.0 - (1.0 - math.log((i + 2) / (i + 1)) / math.log(rows)) ** updates for i in range(rows - 1))
    return {"bytes": (updates + 2 * hit) * width * size + 8 * updates, "flops": float(updates * width)}


def tolerance(case):
    # About four times what the path shows against itself in 64 bits: the rounding of 16-bit
    # results and intermediates, and the order of fp32 sums where the result is fp32.
    op, dtype = case["op"], case["dtype"]
    if op == "gemm":
        return {"rel": {"fp32": 2e-6, "fp16": 8e-4, "bf16": 7e-3}[case["out"]]}
    if op == "fused":
        return {"rel": {"fp16": 1.2e-3, "bf16": 1e-2}[dtype]}
    if op == "attention":
        return {"rel": {"fp16": 1.5e-3, "bf16": 1.2e-2}[dtype]}
    if op == "decode":
        return {"rel": {"fp16": 8e-4, "bf16": 7e-3}[dtype]}
    # every addition into a row rounds the running value, in whatever order they come: the error of a
    # row grows with the root of its additions (measured: 1.7e-3 in bf16 for one a row, 2.9e-2 for 273)
    return {"rel": {"fp32": 1.2e-7, "fp16": 8e-4, "bf16": 7e-3}[dtype] * max(1.0, math.sqrt(case["updates"] / case["rows"]))}
