"""The work that a program using tallax_amd has it do, as cases that can be timed and compared.

Each case is one public call (or the two calls of one step) on inputs that
live on the GPU: exact and approximate top-k, the fused sampler and its wide
form, row sorts with and without a gather, cumulative sums and the prefill
pipeline.  `listed()` holds the shapes that stand for each use, `draw()` more
of the same ranges, odd and ragged sizes, data types and options among them.
"""
from __future__ import annotations

import math

import torch

from tallax_amd import prefill, sampling, tax, tumpy

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "i32": torch.int32}
SIZES = {"f32": 4, "bf16": 2, "i32": 4}
BLOCK_TOKEN, NUM_BINS = 8, 128  # top_dynamic_k's defaults


def listed():
    return [
        # a few rows of a mid-sized score table: one call's latency
        {"name": "topk_few_rows", "op": "topk", "rows": 8, "cols": 32768, "k": 64, "dtype": "f32"},
        # candidates of a decode batch over a whole vocabulary, with log-probabilities kept in float32
        {"name": "topk_vocab", "op": "topk", "rows": 128, "cols": 151936, "k": 50, "dtype": "f32"},
        # a mixture-of-experts router: every token of a prefill chunk picks 8 of 128 experts
        {"name": "topk_router", "op": "topk", "rows": 65536, "cols": 128, "k": 8, "dtype": "f32"},
        # the approximate top-k of the same decode batch, automatic schedule
        {"name": "topk_approx", "op": "approx", "rows": 128, "cols": 151936, "k": 50, "dtype": "f32"},
        # one user's next token: the smallest call of a serving loop
        {"name": "sample_one", "op": "sample", "rows": 1, "cols": 128256, "dtype": "bf16", "masked": False},
        # a decode batch's next tokens: the ordinary call of a serving loop
        {"name": "sample_decode", "op": "sample", "rows": 256, "cols": 128256, "dtype": "bf16", "masked": False},
        # constrained decoding on float32 logits of an odd vocabulary: most tokens are -inf, no row is aligned
        {"name": "sample_masked", "op": "sample", "rows": 67, "cols": 151937, "dtype": "f32", "masked": True},
        # a decode batch whose requests ask for top_k up to 1024
        {"name": "sample_wide", "op": "wide", "rows": 256, "cols": 128256, "dtype": "bf16", "max_k": 1024},
        # stable argsort of short keys and the gather of their payload
        {"name": "argsort_gather", "op": "argsort_gather", "rows": 256, "cols": 4096, "dtype": "bf16"},
        # a whole vocabulary's probabilities in descending order with their tokens, for a prefill's rows: the largest
        {"name": "sort_vocab", "op": "sort", "rows": 1024, "cols": 201088, "dtype": "f32", "descending": True,
         "argsort": True, "keys": 1, "payload": 0},
        # softmax, top 2048, cumulative sum and top-p cutoff of a prefill's rows
        {"name": "prefill", "op": "prefill", "rows": 1024, "cols": 201088, "k": 2048, "p": 0.9},
        # cumulative probabilities over an odd vocabulary
        {"name": "cumsum_vocab", "op": "cumsum", "rows": 64, "cols": 128257, "dtype": "f32", "axis": 1,
         "reverse": False},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cols(rng, lo, hi):
    """A row length: two in three as they fall (odd ones among them), the rest whole multiples of 128."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.67 or n < 256 else n // 128 * 128


def draw(rng):
    op = rng.choice(["topk", "topk", "sample", "sample", "approx", "wide", "sort", "sort", "argsort_gather", "cumsum",
                     "prefill"])
    if op == "topk":
        cols = _cols(rng, 64, 262144)
        return {"op": op, "rows": _log(rng, 1, min(65536, (1 << 25) // cols)), "cols": cols,
                "k": min(cols, rng.choice([1, 2, 8, 50, 64, 128, rng.randint(1, 128)])),
                "dtype": rng.choice(["f32", "f32", "bf16"])}
    if op == "approx":
        cols = _cols(rng, 8192, 262144)
        rows = BLOCK_TOKEN * _log(rng, 1, min(64, (1 << 25) // cols // BLOCK_TOKEN))
        return {"op": op, "rows": rows, "cols": cols, "k": rng.choice([20, 50, 64, 128]),
                "dtype": rng.choice(["f32", "bf16"])}
    if op == "sample":
        cols = _cols(rng, 4096, 262144)
        return {"op": op, "rows": _log(rng, 1, min(1024, (1 << 26) // cols)), "cols": cols,
                "dtype": rng.choice(["bf16", "bf16", "f32"]), "masked": rng.random() < 0.25}
    if op == "wide":
        cols = _cols(rng, 16384, 155648)
        return {"op": op, "rows": _log(rng, 1, 512), "cols": cols, "dtype": rng.choice(["bf16", "bf16", "f32"]),
                "max_k": rng.choice([256, 512, 1024])}
    if op == "sort":
        cols = _cols(rng, 16, 262144)
        return {"op": op, "rows": _log(rng, 1, min(65536, (1 << 24) // cols)), "cols": cols,
                "dtype": rng.choice(["f32", "f32", "bf16", "i32"]), "descending": rng.random() < 0.5,
                "argsort": rng.random() < 0.6, "keys": rng.choice([1, 1, 1, 2]), "payload": rng.choice([0, 0, 1])}
    if op == "argsort_gather":
        cols = _cols(rng, 256, 16384)
        return {"op": op, "rows": _log(rng, 1, min(4096, (1 << 24) // cols)), "cols": cols,
                "dtype": rng.choice(["bf16", "f32"])}
    if op == "cumsum":
        line = _cols(rng, 128, 262144)
        lines = _log(rng, 1, min(4096, (1 << 25) // line))
        axis = rng.choice([0, 1, 1, 1])
        return {"op": op, "rows": line if axis == 0 else lines, "cols": lines if axis == 0 else line,
                "dtype": rng.choice(["f32", "f32", "i32"]), "axis": axis, "reverse": rng.random() < 0.25}
    cols = _cols(rng, 8192, 262144)
    return {"op": op, "rows": _log(rng, 1, min(1024, (1 << 27) // cols)), "cols": cols,
            "k": rng.choice([256, 1024, 2048, rng.randint(256, 2048)]), "p": rng.choice([0.5, 0.9, 0.95])}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, rows, cols, dtype, scale):
    return (torch.randn((rows, cols), generator=g, device="cuda") * scale).to(DTYPES[dtype])


def _operand(g, rows, cols, dtype):
    """A sort operand: normal floats, or whole numbers with some ties."""
    if dtype == "i32":
        return torch.randint(-(1 << 20), 1 << 20, (rows, cols), generator=g, device="cuda", dtype=torch.int32)
    return _normal(g, rows, cols, dtype, 1.0)


def prepare(case, seed):
    g = _gen(seed)
    op, rows, cols = case["op"], case["rows"], case["cols"]
    s = {"case": case}
    if op in ("topk", "approx"):
        s["x"] = _normal(g, rows, cols, case["dtype"], 2.0)
    elif op in ("sample", "wide"):
        x = torch.randn((rows, cols), generator=g, device="cuda") * 3.0
        if case.get("masked"):
            # three rows in four keep some 1 to 600 tokens, the fourth keeps all
            share = torch.randint(1, 601, (rows, 1), generator=g, device="cuda").float() / cols
            keep = torch.rand((rows, cols), generator=g, device="cuda") < share
            keep[3::4] = True
            keep[:, 0] = True
            x = x.masked_fill(~keep, float("-inf"))
        s["x"] = x.to(DTYPES[case["dtype"]])
        # a request's own settings, as a serving loop keeps them on the GPU
        s["meta"] = sampling.SamplingMetadata(
            torch.randint(1, 1025, (rows,), generator=g, device="cuda", dtype=torch.int32),
            torch.rand((rows,), generator=g, device="cuda") * 0.3 + 0.7,
            torch.rand((rows,), generator=g, device="cuda") + 0.5)
        s["key"] = torch.randint(0, 1 << 30, (2,), generator=g, device="cuda", dtype=torch.int32)
    elif op == "sort":
        if case["descending"] and case["dtype"] == "f32" and case["keys"] == 1:
            # probabilities: what is sorted downwards in earnest
            s["x"] = [torch.softmax(_normal(g, rows, cols, "f32", 2.0), dim=1)]
        elif case["keys"] == 2:
            # a coarse first key, so that the second one decides
            s["x"] = [torch.randint(0, 64, (rows, cols), generator=g, device="cuda", dtype=torch.int32),
                      _operand(g, rows, cols, case["dtype"])]
        else:
            s["x"] = [_operand(g, rows, cols, case["dtype"])]
        s["x"] += [_normal(g, rows, cols, "f32", 1.0) for _ in range(case["payload"])]
    elif op == "argsort_gather":
        # keys on a grid of sixteenths, so that the stable order matters
        x = torch.randn((rows, cols), generator=g, device="cuda") * 16
        s["x"] = (x.round() / 16).to(DTYPES[case["dtype"]])
        s["v"] = _normal(g, rows, cols, "f32", 1.0)
    elif op == "cumsum":
        if case["dtype"] == "i32":
            s["x"] = torch.randint(0, 1000, (rows, cols), generator=g, device="cuda", dtype=torch.int32)
        else:
            s["x"] = torch.softmax(_normal(g, rows, cols, "f32", 2.0), dim=case["axis"])
    else:
        # peaked logits, of which some hundred tokens hold nine tenths
        s["x"] = _normal(g, rows, cols, "f32", 4.0)
    return s


def run(state):
    c, x = state["case"], state["x"]
    op = c["op"]
    if op == "topk":
        return tax.top_k(x, c["k"])
    if op == "approx":
        return tax.top_dynamic_k(x, c["k"], c["k"])
    if op == "sample":
        return sampling.sample(state["key"], x, state["meta"])
    if op == "wide":
        return sampling.sample(state["key"], x, state["meta"], max_k=c["max_k"])
    if op == "sort":
        return tax.sort(x, num_keys=c["keys"], descending=c["descending"], return_argsort=c["argsort"])
    if op == "argsort_gather":
        order = tumpy.argsort(x)
        return order, tumpy.take_along_axis(state["v"], order, 1)
    if op == "cumsum":
        return tax.cumsum(x, c["axis"], c["reverse"])
    return prefill.softmax_topk_cumsum(x, c["k"], c["p"])


def work(case):
    op, n = case["op"], case["rows"] * case["cols"]
    size = SIZES[case.get("dtype", "f32")]
    rows = case["rows"]
    if op == "topk":
        return {"bytes": n * size + rows * case["k"] * (size + 4), "flops": 0}
    if op == "approx":
        return {"bytes": n * size + rows * case["k"] * (size + 4) + rows * 8, "flops": 0}
    if op in ("sample", "wide"):
        return {"bytes": n * size + rows * 16 + 8, "flops": 0}
    if op == "sort":
        first = 4 if case["keys"] == 2 else size
        keys = first if case["keys"] == 1 else first + size
        return {"bytes": n * (2 * keys + 8 * case["payload"] + 4 * case["argsort"]), "flops": 0}
    if op == "argsort_gather":
        return {"bytes": n * (size + 4 + 4 + 4), "flops": 0}
    if op == "cumsum":
        return {"bytes": 2 * n * size, "flops": n}
    return {"bytes": n * 4 + rows * (12 * case["k"] + 4), "flops": 3 * n}


def tolerance(case):
    if case["op"] == "cumsum" and case["dtype"] == "f32":
        # sums of up to 262144 probabilities: 4.4e-7 from 64 bits at [64, 128257], more on longer lines
        return {"rel": 4e-6}
    if case["op"] == "prefill":
        # float32 exponentials and sums: 1.1e-7 from 64 bits; a cutoff moves by one where the sum meets p
        # within rounding
        return {"rel": 1e-6, "differ": 0.005}
    return "exact"


def exact(case, seed):
    op = case["op"]
    if op in ("sample", "wide"):
        return None  # tokens: whole numbers
    s = prepare(case, seed)
    x = s["x"]
    if op in ("topk", "approx"):
        v, i = torch.sort(x.double(), dim=1, descending=True, stable=True)
        v, i = v[:, :case["k"]], i[:, :case["k"]]
        return (v, i.int()) if op == "topk" else (v, None, None, None, None)
    if op == "sort":
        if case["keys"] == 2 or case["dtype"] == "i32":
            return None  # whole numbers, and floats that are only moved
        v, i = torch.sort(x[0].double(), dim=1, descending=case["descending"], stable=True)
        outs = [v] + [p.double().gather(1, i) for p in x[1:]]
        return tuple(outs + ([None] if case["argsort"] else []))
    if op == "argsort_gather":
        i = torch.sort(x.double(), dim=1, stable=True)[1]
        return None, s["v"].double().gather(1, i)
    if op == "cumsum":
        if case["dtype"] == "i32":
            return None
        y = x.double()
        if case["reverse"]:
            return y.flip(case["axis"]).cumsum(case["axis"]).flip(case["axis"])
        return y.cumsum(case["axis"])
    probs, sums = [], []
    for part in x.split(128):
        e = torch.softmax(part.double(), dim=1)
        top = torch.sort(e, dim=1, descending=True)[0][:, :case["k"]]
        probs.append(top)
        sums.append(top.cumsum(1))
    return torch.cat(probs), None, torch.cat(sums), None
