"""Timed cases of the attention forward: what programs have `flash_attention_runtime.forward` do.

A case is one call on Q, K, V of shape [B, H, N, D] that are already on the GPU:

  B, H, N, D   batch, heads, sequence length, head dim (64 or 128)
  dtype        "fp16" or "bf16"
  causal       lower-triangular mask
  lse          also return the logsumexp (what a training step keeps for its backward pass)
  layout       "bhnd": contiguous tensors; "bnhd": views of [B, N, H, D] tensors, as a projection
               leaves them (the output then has that layout too)
  sigma        standard deviation of Q and K (1, or 3: scores so wide that a few keys decide a row)
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "flash-attention_amd"))

import flash_attention_runtime as fa  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, B, H, N, D, dtype, causal, lse=False, layout="bhnd", sigma=1.0):
    return {"name": name, "B": B, "H": H, "N": N, "D": D, "dtype": dtype, "causal": causal,
            "lse": lse, "layout": layout, "sigma": sigma}


def listed():
    return [
        # One short prompt with few heads: the latency of a call, its launch and its allocation.
        _case("tiny", 1, 2, 128, 64, "fp16", False, lse=True),
        # A batch of short encoder sequences that no tile divides, straight from the projections.
        _case("short-ragged", 16, 16, 200, 64, "fp16", False, layout="bnhd"),
        # A training step on short causal sequences; the backward pass needs the logsumexp.
        _case("short-causal-train", 4, 32, 512, 128, "bf16", True, lse=True),
        # The benchmark's D = 64 configuration: an encoder layer at an ordinary length.
        _case("encoder-d64", 4, 16, 1024, 64, "fp16", False),
        # A causal training batch whose length is no power of two, from the projections.
        _case("causal-d64-train", 4, 16, 1000, 64, "bf16", True, lse=True, layout="bnhd"),
        # The benchmark's ragged configuration: one prompt of 3000 tokens, wide scores.
        _case("prompt-ragged", 1, 16, 3000, 128, "fp16", True, sigma=3.0),
        # A long prompt on a rank that holds few heads (heads split over devices).
        _case("long-few-heads", 1, 2, 8192, 128, "bf16", True),
        # A small model's encoder: few heads and too few q-tiles to fill the GPU.
        _case("encoder-few-heads", 2, 4, 2048, 64, "fp16", False),
        # The D = 64 row of the comparison with torch: a large batch at 4096.
        _case("batch-d64", 4, 32, 4096, 64, "fp16", False),
        # The headline configuration of the benchmark.
        _case("batch-4096", 4, 32, 4096, 128, "fp16", False),
        # The benchmark's causal bf16 configuration as a training step runs it.
        _case("train-8192", 2, 32, 8192, 128, "bf16", True, lse=True),
        # The benchmark's longest configuration: one prompt of 16384 tokens, wide scores.
        _case("prompt-16384", 1, 16, 16384, 128, "fp16", True, sigma=3.0),
    ]


def _pairs(case):
    """Query-key pairs of one head that the mask leaves."""
    n = case["N"]
    return n * (n + 1) // 2 if case["causal"] else n * n


def _flops(case):
    return 4.0 * case["B"] * case["H"] * _pairs(case) * case["D"]


def draw(rng):
    """Lengths from 100 to 16384 and batches from 1 to 16, spread over their logarithm, with 1 to
    256 heads in the whole call and at most a third of the largest listed case's products."""
    while True:
        n = int(round(math.exp(rng.uniform(math.log(100), math.log(16384)))))
        if rng.random() < 0.4:
            n = max(128, n // 128 * 128)
        heads = rng.choice([1, 2, 4, 6, 8, 12, 16, 20, 32, 40])
        case = {"B": int(round(math.exp(rng.uniform(0.0, math.log(16))))), "H": heads, "N": n,
                "D": rng.choice([64, 128]), "dtype": rng.choice(["fp16", "bf16"]),
                "causal": rng.random() < 0.5, "lse": rng.random() < 0.4,
                "layout": "bnhd" if rng.random() < 0.4 else "bhnd",
                "sigma": 3.0 if rng.random() < 0.25 else 1.0}
        if case["B"] * heads <= 256 and _flops(case) <= 3.7e11:
            return case


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    b, h, n, d = case["B"], case["H"], case["N"], case["D"]
    shape = (b, n, h, d) if case["layout"] == "bnhd" else (b, h, n, d)
    out = []
    for sigma in (case["sigma"], case["sigma"], 1.0):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        x = (x * sigma).to(_DTYPES[case["dtype"]])
        out.append(x.permute(0, 2, 1, 3) if case["layout"] == "bnhd" else x)
    return out


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    return {"q": q, "k": k, "v": v, "causal": case["causal"], "lse": case["lse"]}


def run(state):
    return fa.forward(state["q"], state["k"], state["v"], causal=state["causal"],
                      return_lse=state["lse"])


def work(case):
    elems = case["B"] * case["H"] * case["N"]
    return {"bytes": elems * (4 * 2 * case["D"] + (4 if case["lse"] else 0)),
            "flops": _flops(case)}


def tolerance(case):
    # P and O are rounded to the input type (unit roundoff 2^-11 and 2^-8): about four times the
    # error against 64 bits that the forward shows (fp16 2.9e-4, bf16 2.1e-3), which is also what
    # a correct forward with its sums in another order shows.
    return {"rel": 1.2e-3} if case["dtype"] == "fp16" else {"rel": 8.5e-3}


def exact(case, seed):
    """softmax(Q K^T / sqrt(D) [+ mask]) V and its logsumexp in 64 bits, by blocks of rows."""
    q, k, v = _inputs(case, seed)
    b, h, n, d = case["B"], case["H"], case["N"], case["D"]
    o = torch.empty_like(q, dtype=torch.float64)
    lse = torch.empty((b, h, n), dtype=torch.float64, device="cuda")
    cols = torch.arange(n, device="cuda")
    rows = max(1, min(n, (1 << 25) // n))
    for i in range(b):
        for j in range(h):
            kt = k[i, j].double().t().contiguous()
            vd = v[i, j].double().contiguous()
            for r in range(0, n, rows):
                e = min(n, r + rows)
                s = torch.mm(q[i, j, r:e].double().contiguous(), kt) / math.sqrt(d)
                if case["causal"]:
                    s.masked_fill_(cols[None, :] > cols[r:e, None], -math.inf)
                m = s.amax(dim=1, keepdim=True)
                p = torch.exp(s - m)
                t = p.sum(dim=1, keepdim=True)
                o[i, j, r:e] = torch.mm(p, vd) / t
                lse[i, j, r:e] = (m + torch.log(t))[:, 0]
    return (o, lse) if case["lse"] else o
