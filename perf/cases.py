"""The work a user has this framework do, as cases that can be timed: single and batched sparse int4 products, products
routed over many resident deltas, LoRA adapters beside them, and the packing of a delta, each through the op a serving or
conversion program calls (`triteia_amd.python.ops`).

A case is a dict of plain values.  `op` names the call; k and m are the layer's input and output widths, `n` the number of
resident matrices (or deltas), `tokens` the rows of activations (per matrix for `bmm`), `routing` how tokens choose among
them, `base` whether the layer's dense fp16 weight is part of the call, `adapters` / `rank` the LoRA side, `dtype` the
activations' element type.
"""
import math

import numpy as np
import torch

from triteia_amd.python import ops
from triteia_amd.python.ops.utils.generator import fp16_to_sparse
from triteia_amd.workloads import random_activations, random_packed_deltas, uniform_indices, zipf_indices

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(op, k, m, tokens=0, n=1, routing="", base=False, adapters=0, rank=0, dtype="fp16"):
    return {"op": op, "k": k, "m": m, "tokens": tokens, "n": n, "routing": routing, "base": base,
            "adapters": adapters, "rank": rank, "dtype": dtype}


def listed():
    cases = {
        # one request being decoded on one compressed layer: the smallest call there is
        "matmul_decode": _case("matmul", 4096, 4096, tokens=1),
        # a handful of requests of an odd number on the long side of an MLP (few columns, long k)
        "matmul_ragged": _case("matmul", 11008, 4096, tokens=37),
        # the prompt of one model, not a whole number of tiles
        "matmul_prefill": _case("matmul", 4096, 11008, tokens=4000),
        # eight models with one request each, one token per model
        "bmm_decode": _case("bmm", 4096, 4096, tokens=1, n=8),
        # the framework's headline: a decode batch routed evenly over sixteen variants of one layer
        "sbmm_decode": _case("sbmm", 4096, 4096, tokens=64, n=16, routing="uniform"),
        # a small decode batch spread thinly over many variants, with the base model's weight
        "sbmm_sparse_base": _case("sbmm", 11008, 4096, tokens=13, n=32, routing="uniform", base=True),
        # prompts and decodes of several popular variants in one batch
        "sbmm_mixed": _case("sbmm", 4096, 11008, tokens=1000, n=32, routing="zipf:1.2"),
        # the largest layer and the most resident variants
        "sbmm_large": _case("sbmm", 8192, 28672, tokens=256, n=64, routing="zipf:1.2"),
        # one layer with its base weight, LoRA adapters and compressed variants in one batch
        "ldmm": _case("ldmm", 4096, 11008, tokens=256, n=32, routing="zipf:1.5", base=True, adapters=32, rank=16),
        # adapters alone, any order of requests, by the per-token op
        "lora_decode": _case("bgmv", 4096, 11008, tokens=100, routing="zipf:1.2", adapters=32, rank=16),
        # adapters alone on prompts, requests grouped by adapter, in bf16
        "lora_prefill": _case("sgmv", 4096, 4096, tokens=1000, routing="uniform", adapters=8, rank=64, dtype="bf16"),
        # a dense variant being quantised and packed when it is loaded
        "pack": _case("pack", 4096, 4096),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo=512, hi=13824):
    """A layer width: any multiple of 128, spread over its logarithm."""
    return max(lo, min(hi, 128 * _log_int(rng, lo / 128, hi / 128)))


def _routing(rng):
    return rng.choice(["uniform", "zipf:1.2", "zipf:1.5"])


def draw(rng):
    most = [work(c) for c in listed()]
    most_flops, most_bytes = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    op = rng.choice(["matmul", "matmul", "bmm", "sbmm", "sbmm", "sbmm", "ldmm", "bgmv", "sgmv", "pack"])
    k, m = _width(rng), _width(rng)
    if op == "matmul":
        c = _case(op, k, m, tokens=_log_int(rng, 1, 4096))
    elif op == "bmm":
        c = _case(op, k, m, tokens=_log_int(rng, 1, 64), n=_log_int(rng, 2, 32))
    elif op == "sbmm":
        c = _case(op, k, m, tokens=_log_int(rng, 1, 4096), n=_log_int(rng, 2, 64), routing=_routing(rng), base=rng.random() < 0.3)
    elif op == "ldmm":
        c = _case(op, k, m, tokens=_log_int(rng, 8, 1024), n=_log_int(rng, 2, 32), routing=_routing(rng), base=rng.random() < 0.7,
                  adapters=_log_int(rng, 2, 32), rank=rng.choice([8, 16, 32, 64]))
    elif op in ("bgmv", "sgmv"):
        c = _case(op, k, m, tokens=_log_int(rng, 1, 256 if op == "bgmv" else 2048), routing=_routing(rng), adapters=_log_int(rng, 2, 64),
                  rank=rng.choice([8, 16, 32, 64, 128]), dtype=rng.choice(["fp16", "bf16"]))
    else:
        c = _case(op, min(k, 4096), min(m, 4096))
    while c["tokens"] > 1 and (work(c)["flops"] > most_flops or work(c)["bytes"] > most_bytes):
        c["tokens"] //= 2
    return c


def _indices(routing, tokens, n, seed):
    """Per token: one of n, or -1 (no variant)."""
    if routing == "uniform":
        return uniform_indices(tokens, n, seed)
    return zipf_indices(tokens, n, float(routing.split(":")[1]), seed, frac_none=0.1)


def _dense(rows, columns, seed, dtype, spread):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((rows, columns), generator=g, device="cuda") * spread).to(dtype)


def prepare(case, seed):
    op, k, m, tokens, n, adapters, rank = (case[f] for f in ("op", "k", "m", "tokens", "n", "adapters", "rank"))
    dtype = _DTYPES[case["dtype"]]
    s = {"op": op}
    if op == "pack":
        s["weight"] = _dense(k, m, seed, torch.float16, 0.02)
        s["scale"] = (s["weight"].abs().amax(0, keepdim=True) * (2 / 15)).contiguous()   # the largest weight of a column is 7.5 steps
        return s
    rows = tokens * n if op == "bmm" else tokens
    s["x"] = random_activations(rows, k, seed + 1, "cuda").to(dtype)
    if op in ("matmul", "bmm", "sbmm", "ldmm"):
        s["qweight"], s["meta"], s["scales"] = random_packed_deltas(n, k, m, seed + 2, "cuda")
    if op == "bmm":
        s["x"] = s["x"].view(n, tokens, k)
    if adapters:
        s["A"] = _dense(adapters * k, rank, seed + 3, dtype, 0.02).view(adapters, k, rank)
        s["B"] = _dense(adapters * rank, m, seed + 4, dtype, 0.02).view(adapters, rank, m)
    if op in ("sbmm", "ldmm"):
        s["base"] = _dense(m, k, seed + 5, dtype, 0.02) if case["base"] else None
    if case["routing"]:
        index = _indices(case["routing"], tokens, adapters if op in ("bgmv", "sgmv") else n, seed + 6)
        if op == "ldmm":
            # a routed token takes an adapter or a compressed variant; adapters come first in the op's index space
            coin = np.random.default_rng(seed + 7).random(tokens) < 0.5
            index = np.where((index >= 0) & coin, index % adapters, np.where(index >= 0, index + adapters, -1))
        if op == "sgmv":
            index = np.sort(index)   # this op takes requests grouped by adapter
        s["indices"] = torch.from_numpy(index.astype(np.int32)).cuda()
    return s


def run(s):
    op = s["op"]
    if op == "matmul":
        return ops.matmul_4bit_2_4(s["qweight"][0], s["x"], s["meta"][0], s["scales"][0])
    if op == "bmm":
        return ops.bmm_4bit_2_4(s["qweight"], s["x"], s["meta"], s["scales"])
    if op == "sbmm":
        return ops.sbmm_4bit_2_4_native(s["qweight"], s["x"], s["meta"], s["scales"], s["indices"], base_weight=s["base"])
    if op == "ldmm":
        return ops.ldmm(s["indices"], s["x"], s["A"], s["B"], s["qweight"], s["meta"], s["scales"], base_weight=s["base"])
    if op == "bgmv":
        return ops.lora_bgmv(s["A"], s["B"], s["x"], s["indices"])
    if op == "sgmv":
        return ops.lora_sgmv(s["A"], s["B"], s["x"], s["indices"])
    _, qweight, scales, meta, meta_raw = fp16_to_sparse(s["weight"], s["scale"])
    return {"qweight": qweight, "scales": scales, "meta": meta, "meta_raw": meta_raw}


def _expected_distinct(routing, tokens, n):
    """How many of n are in use by a batch on average, and the share of its tokens that take one."""
    if routing == "uniform":
        p = np.full(n, 1.0 / (n + 1))
    else:
        p = np.arange(1, n + 1, dtype=np.float64) ** -float(routing.split(":")[1])
        p *= 0.9 / p.sum()
    return float((1.0 - (1.0 - p) ** tokens).sum()), float(p.sum())


def work(case):
    """Bytes: every weight in use, the activations and the output once; operations: 2 per weight of the dense layer
    and token (LoRA: of the two thin matrices)."""
    op, k, m, tokens, n, adapters, rank = (case[f] for f in ("op", "k", "m", "tokens", "n", "adapters", "rank"))
    packed = k * m * 0.375 + 2 * m
    if op == "pack":
        return {"bytes": 2.0 * k * m + 2 * m + packed + k * m / 8, "flops": 0.0}
    if op == "matmul":
        return {"bytes": packed + 2.0 * tokens * (k + m), "flops": 2.0 * tokens * k * m}
    if op == "bmm":
        return {"bytes": n * (packed + 2.0 * tokens * (k + m)), "flops": 2.0 * n * tokens * k * m}
    bytes_, flops = 2.0 * tokens * (k + m) + 4.0 * tokens, 0.0
    if case["base"]:
        bytes_ += 2.0 * k * m
        flops += 2.0 * tokens * k * m
    routed = adapters if op in ("bgmv", "sgmv") else n
    delta_tokens, lora_tokens = {"sbmm": (tokens, 0), "ldmm": (tokens / 2, tokens / 2)}.get(op, (0, tokens))
    if delta_tokens:
        distinct, share = _expected_distinct(case["routing"], delta_tokens, n)
        bytes_ += distinct * packed
        flops += 2.0 * delta_tokens * share * k * m
    if lora_tokens:
        distinct, share = _expected_distinct(case["routing"], lora_tokens, routed)
        bytes_ += min(distinct, adapters) * 2.0 * rank * (k + m)
        flops += 2.0 * lora_tokens * share * rank * (k + m)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Four times what the ops show against the same product in 64 bits (rounding of the stored results included)."""
    if case["op"] == "pack":
        return "exact"
    return {"rel": 1e-2, "max": 5e-2} if case["dtype"] == "bf16" else {"rel": 1e-3, "max": 6e-3}
