"""Workloads that stand for what users of `flash_colsum` run, for timing and for comparing outputs.

The operator reduces a pair of attention operands to one importance value per key position.  Its users
rank the tokens of an encoder (vision or text, whole batches at a time, `cls_len` where only the class
token's attention counts) or the key cache of a decoder (the last window of queries against a long
context, the prompt against itself, grouped key heads), and keep the top k.  The cases cover those calls
from a few microseconds of work to half a gigabyte of keys: `listed()` names twelve of them, `draw()` makes
more of the same five families.

A case is a dict of plain values:
  family      which of the five families below it belongs to
  batch, heads, kv_heads, q_len, k_len, head_dim
  dtype       "fp16", "bf16" or "fp32" operands
  layout      "heads": dense (B, H, S, D); "tokens": the (B, S, H, D) storage that a projection leaves
              behind, seen through a transpose
  cls_len     average over the first rows only (0: over all of them)
  top_k       return the k most attended positions instead of the means (0: the means)
  spread      standard deviation of the keys' common part of the logits: 0 gives every key a similar
              mean, 1 or 2 the heavy hitters of a decoder's cache
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-colsum_amd"))

from flash_colsum import flash_colsum, flash_colsum_f32, flash_colsum_topk  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, family, batch, heads, q_len, k_len, head_dim, dtype="fp16", kv_heads=None, layout="heads", cls_len=0, top_k=0, spread=0.0):
    c = {"family": family, "batch": batch, "heads": heads, "kv_heads": kv_heads or heads, "q_len": q_len, "k_len": k_len, "head_dim": head_dim,
         "dtype": dtype, "layout": layout, "cls_len": cls_len, "top_k": top_k, "spread": spread}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short text through one small layer: launches and the host path are all there is
        _case("encoder_small", "encoder", 2, 4, 512, 512, 64),
        # the batched self-attention shape that the benchmark quotes: 2048 tokens, a batch of 8
        _case("encoder_s2048", "encoder", 8, 16, 2048, 2048, 64),
        # a batch of the batched sweep in bf16, as a model trained in bf16 hands it over
        _case("encoder_s1024_bf16", "encoder", 64, 16, 1024, 1024, 64, dtype="bf16", layout="tokens"),
        # 128-wide heads at ordinary length
        _case("encoder_d128_bf16", "encoder", 8, 16, 1024, 1024, 128, dtype="bf16"),
        # vision encoder, 14 x 14 patches and a class token, as the projection stores it
        _case("vision_s197", "encoder", 64, 12, 197, 197, 64, layout="tokens"),
        # vision encoder, 24 x 24 patches and a class token: only the class token's row is averaged
        _case("vision_s577_cls", "encoder", 32, 16, 577, 577, 64, cls_len=1),
        # the same encoder run in fp32, all rows
        _case("vision_s577_fp32", "encoder", 16, 16, 577, 577, 64, dtype="fp32"),
        # a long document, one sequence: more keys than a workgroup holds
        _case("document_s8192", "document", 1, 16, 8192, 8192, 64),
        # the last 128 queries of a decoder against its cache
        _case("window_q128_k16384", "window", 1, 32, 128, 16384, 128, spread=1.0),
        # long context: 512 queries against 65536 keys, half a gigabyte of them
        _case("window_q512_k65536", "window", 1, 32, 512, 65536, 128, spread=1.0),
        # a prompt against itself, causal, in bf16
        _case("prompt_s4096_bf16", "prompt", 1, 32, 4096, 4096, 128, dtype="bf16", spread=1.0),
        # cache pruning of a decoder with grouped key heads: the 1024 keys that the last 64 queries of each sequence attend to most
        _case("prune_gqa_k8192", "prune", 4, 32, 64, 8192, 128, dtype="bf16", kv_heads=8, top_k=1024, spread=1.5),
    ]


def _log_int(rng, lo, hi):
    """Whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_family(rng):
    family = rng.choice(["encoder", "encoder", "encoder", "document", "window", "prompt", "prune"])
    if family == "encoder":
        s = rng.choice([rng.randint(49, 300), _log_int(rng, 64, 2048), _log_int(rng, 256, 2048)])
        return _case(None, family, _log_int(rng, 1, 128), rng.choice([4, 6, 8, 12, 16]), s, s, rng.choice([64, 64, 64, 64, 128, 128, 32, 80, 96]),
                     dtype=rng.choice(["fp16", "fp16", "bf16", "fp32"]), layout=rng.choice(["heads", "tokens"]),
                     cls_len=rng.choice([0, 0, 0, 0, 1, 4]))
    if family == "document":
        s = _log_int(rng, 2049, 11000)
        return _case(None, family, 1, rng.choice([8, 12, 16]), s, s, rng.choice([64, 64, 128]), dtype=rng.choice(["fp16", "fp16", "bf16"]),
                     layout=rng.choice(["heads", "tokens"]))
    if family == "window":
        return _case(None, family, 1, rng.choice([8, 16, 32]), _log_int(rng, 16, 512), _log_int(rng, 1024, 65536), rng.choice([64, 128, 128]),
                     dtype=rng.choice(["fp16", "fp16", "bf16"]), layout=rng.choice(["heads", "heads", "tokens"]), spread=rng.choice([0.0, 1.0]))
    if family == "prompt":
        s = _log_int(rng, 300, 6000)
        return _case(None, family, 1, rng.choice([8, 16, 32]), s, s, rng.choice([64, 128, 128]), dtype=rng.choice(["fp16", "bf16"]),
                     layout=rng.choice(["heads", "tokens"]), spread=rng.choice([0.0, 1.0]))
    kv_heads = rng.choice([2, 4, 8])
    k_len = _log_int(rng, 1000, 32768)
    return _case(None, family, rng.choice([1, 2, 3, 4, 8]), kv_heads * rng.choice([1, 2, 4, 8]), rng.choice([1, 16, 32, 64, rng.randint(2, 128)]), k_len,
                 rng.choice([64, 128, 128]), dtype=rng.choice(["fp16", "bf16", "bf16"]), kv_heads=kv_heads, top_k=_log_int(rng, 64, min(k_len // 2, 4096)),
                 spread=rng.choice([1.0, 1.5]))


def draw(rng):
    while True:
        c = _draw_family(rng)
        w = work(c)
        # within the largest listed case's work, and for operands that are converted first within what that case takes
        if w["flops"] <= 2.0e11 and w["bytes"] <= (1.2e8 if c["dtype"] == "fp32" else 5.0e8):
            return c


def _rows(case):
    return min(case["cls_len"] or case["q_len"], case["q_len"])


def _causal(case):
    return case["family"] in ("window", "prompt", "prune")


def _operand(gen, batch, heads, seq, dim, case):
    """fp32 N(0, 1) of logical shape (B, H, S, D) in the case's storage order."""
    shape = (batch, seq, heads, dim) if case["layout"] == "tokens" else (batch, heads, seq, dim)
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return x.transpose(1, 2) if case["layout"] == "tokens" else x


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    b, hq, hk, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    q = _operand(gen, b, hq, case["q_len"], d, case)
    k = _operand(gen, b, hk, case["k_len"], d, case)
    if case["spread"]:
        # queries of a key head share a direction, and keys lie along it more or less: their logits get a common part
        # of standard deviation `spread` at the default scale
        u = torch.randn((b, hk, 1, d), generator=gen, device="cuda")
        u = u / u.norm(dim=-1, keepdim=True)
        along = torch.randn((b, 1, case["k_len"], 1), generator=gen, device="cuda")
        q.add_(u.repeat_interleave(hq // hk, dim=1), alpha=d ** 0.25)
        k.add_(along * u, alpha=case["spread"] * d ** 0.25)
    dtype = _DTYPES[case["dtype"]]
    return dict(case=case, q=q.to(dtype), k=k.to(dtype))


def run(state):
    case, q, k = state["case"], state["q"], state["k"]
    if case["top_k"]:
        return flash_colsum_topk(q, k, case["top_k"], is_causal=True, extended=True)
    if _causal(case):
        # means of a long context are below fp16's normal range: taken as fp32
        return flash_colsum_f32(q, k, is_causal=True)
    return flash_colsum(q, k, cls_len=case["cls_len"] or None)


def work(case):
    """One read of the averaged queries and of the keys, one write of the result; one Q K^T over the visible pairs."""
    b, hq, hk, d, n_k, rows = case["batch"], case["heads"], case["kv_heads"], case["head_dim"], case["k_len"], _rows(case)
    size = 4 if case["dtype"] == "fp32" else 2
    pairs = rows * n_k
    if _causal(case):
        past = max(0, n_k - case["q_len"])
        pairs = sum(min(n_k, past + i + 1) for i in range(rows))
    out = case["top_k"] * 12 if case["top_k"] else n_k * (4 if _causal(case) else 2)
    return {"bytes": size * b * d * (hq * rows + hk * n_k) + b * out, "flops": 2 * b * hq * d * pairs}


def tolerance(case):
    """About four times the distance from a float64 evaluation of the same operands that was measured on an MI355X."""
    if case["top_k"]:
        # fp32 means: 9e-7 at most; neighbours of the sorted selection whose means are that close may trade places
        return {"rel": 3e-6, "max": 4e-6, "differ": 0.004}
    if _causal(case):
        if case["dtype"] == "fp16" and case["head_dim"] == 64:
            return {"rel": 2e-5, "max": 6e-5}  # scores from an operand that is scaled, then rounded to fp16: 4e-6 and 1.2e-5
        return {"rel": 3e-6, "max": 4e-6}  # fp32 sums: 7e-7 and 9e-7 at most
    # a mean rounded to fp16: up to 7e-5 (2e-4 for fp32 operands, which are rounded to fp16 first), single values one unit
    # in the last place (9.8e-4) apart
    return {"rel": 8e-4 if case["dtype"] == "fp32" else 3e-4, "max": 4e-3}
