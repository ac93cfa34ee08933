"""What a user of the attention forward calls it for, and over which sizes.

Every case is one call of `attention(q, k, v, causal, sm_scale)` (with the row
LSE where the caller keeps it), on tensors that are already on the GPU.  The
listed cases are this repository's measured workloads and evaluator shapes,
and generic ones between them; draw() gives more calls of the same ranges.
"""

from __future__ import annotations

import math

import torch

from flash_attn_npu_amd import flash_attention_forward as fa

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, B, H, S, D, dtype, causal, lse=True, layout="bhsd", v="same", dist="normal"):
    """layout "bhsd": dense [B, H, S, D]; "bshd": the [B, S, H, D] output of a
    projection, viewed as [B, H, S, D].  v "e5m2": V in float8_e5m2."""
    c = dict(B=B, H=H, S=S, D=D, dtype=dtype, causal=causal, lse=lse, layout=layout, v=v, dist=dist)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One short sequence, few heads: the latency of a call and of its launch.
        _case("small-b1h8s512d64", 1, 8, 512, 64, "fp16", False, lse=False),
        # A batch of short prompts (an evaluator shape): many heads of a few tiles.
        _case("short-b4h32s256d128", 4, 32, 256, 128, "fp16", True, lse=False),
        # The prompt of one user, its q, k, v as the projections leave them.
        _case("prompt-b1h32s1777d128", 1, 32, 1777, 128, "bf16", True, layout="bshd"),
        # A training or prefill batch at 2048: the headline workload.
        _case("batch-b4h32s2048d128", 4, 32, 2048, 128, "bf16", True),
        # Long context, causal.
        _case("long-b2h16s8192d128", 2, 16, 8192, 128, "bf16", True),
        # An encoder's batch: many heads, D = 64, every key visible.
        _case("encoder-b16h16s1024d64", 16, 16, 1024, 64, "fp16", False),
        # A ragged length with outlying logits: S is no multiple of any tile.
        _case("ragged-b8h32s3000d128", 8, 32, 3000, 128, "bf16", True, dist="outliers"),
        # D = 128 with every key visible (an evaluator shape), inference only.
        _case("full-b4h32s2048d128", 4, 32, 2048, 128, "fp16", False, lse=False),
        # The widest head dim (an evaluator shape).
        _case("wide-b128h8s1024d256", 128, 8, 1024, 256, "bf16", True, lse=False),
        # A narrow head dim at an odd length.
        _case("narrow-b8h16s1500d32", 8, 16, 1500, 32, "fp16", True),
        # One or two heads over a long sequence (a sharded model's slice).
        _case("slice-b1h2s8192d64", 1, 2, 8192, 64, "fp16", False),
        # V stored in fp8 (e5m2).
        _case("fp8v-b2h16s2048d128", 2, 16, 2048, 128, "bf16", True, v="e5m2"),
    ]


def _pairs(c):
    """(query, visible key) pairs of one head."""
    return c["S"] * (c["S"] + 1) // 2 if c["causal"] else c["S"] ** 2


def _cost(c):
    """Grows with a case's time: narrow head dims cost about what D = 64 does."""
    return c["B"] * c["H"] * _pairs(c) * max(c["D"], 64)


def draw(rng):
    """One more call: up to 1024 heads, lengths from 64 to 16384 (most of them odd),
    any head dim, dtype, mask and layout, no dearer than the largest listed case."""
    most = max(_cost(c) for c in listed())
    largest_bytes = max(work(c)["bytes"] for c in listed())
    while True:
        S = int(round(math.exp(rng.uniform(math.log(64), math.log(16384)))))
        heads = math.exp(rng.uniform(0.0, math.log(1024)))
        H = rng.choice([1, 2, 4, 8, 12, 16, 32, 40])
        B = max(1, int(round(heads / H)))
        D = rng.choice([16, 32, 64, 64, 64, 128, 128, 128, 128, 256])
        c = _case(None, B, H, S, D, rng.choice(["fp16", "bf16"]), rng.random() < 0.6, lse=rng.random() < 0.5,
                  layout=rng.choice(["bhsd", "bhsd", "bshd"]), v="e5m2" if rng.random() < 0.1 else "same",
                  dist=rng.choice(["normal", "normal", "normal", "outliers"]))
        if _cost(c) <= most and work(c)["bytes"] <= largest_bytes:
            return c


def _inputs(case, seed):
    """q, k, v from the seed: N(0, 1); "outliers": 1% of the q and k elements 8 times
    larger and v uniform in (-1, 1), as in the ragged workload."""
    g = torch.Generator(device=fa.DEVICE).manual_seed(seed)
    B, H, S, D = (case[k] for k in "BHSD")
    shape = (B, S, H, D) if case["layout"] == "bshd" else (B, H, S, D)
    dtype = DTYPES[case["dtype"]]
    out = []
    for i in range(3):
        if case["dist"] == "outliers" and i == 2:
            t = torch.rand(shape, generator=g, device=fa.DEVICE) * 2.0 - 1.0
        else:
            t = torch.randn(shape, generator=g, device=fa.DEVICE)
            if case["dist"] == "outliers":
                t = torch.where(torch.rand(shape, generator=g, device=fa.DEVICE) < 0.01, t * 8.0, t)
        t = t.to(torch.float8_e5m2 if i == 2 and case["v"] == "e5m2" else dtype)
        out.append(t.permute(0, 2, 1, 3) if case["layout"] == "bshd" else t)
    return out


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    return {"q": q, "k": k, "v": v, "causal": case["causal"], "sm_scale": case["D"] ** -0.5, "lse": case["lse"]}


def run(state):
    return fa.attention(state["q"], state["k"], state["v"], state["causal"], state["sm_scale"],
                        return_lse=state["lse"])


def work(case):
    """q, k, v read once, O (and the LSE, where it is asked for) written once; 2 D
    multiply-adds for each visible pair."""
    rows = case["B"] * case["H"] * case["S"]
    v_bytes = 1 if case["v"] == "e5m2" else 2
    return {"bytes": rows * case["D"] * (6 + v_bytes) + (4 * rows if case["lse"] else 0),
            "flops": 4.0 * case["B"] * case["H"] * _pairs(case) * case["D"]}


def tolerance(case):
    """P and O are rounded to the 16-bit type (bf16 2^-9, fp16 2^-12 relative each) and
    to e5m2 (2^-3) where V has it.  The rounding of P depends on the maximum it is taken
    against, so two orders of the sums differ by about what either is off the exact
    result: measured up to 2.4e-3 (bf16) and 3e-4 (fp16), stated four times that."""
    if case["v"] == "e5m2":
        return {"rel": 0.03, "max": 0.9}
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 0.012}


def exact(case, seed):
    """softmax(q k^T sm_scale) v and its log-sum-exp in float64, by heads and blocks of rows."""
    if case["B"] * case["H"] * _pairs(case) * (2 if case["causal"] else 1) > 2.5e10:
        return None
    q, k, v = _inputs(case, seed)
    B, H, S, D = (case[n] for n in "BHSD")
    o = torch.empty((B, H, S, D), dtype=torch.float64, device=q.device)
    lse = torch.empty((B, H, S), dtype=torch.float64, device=q.device)
    keys = torch.arange(S, device=q.device)
    step = max(1, (1 << 26) // S)  # rows per block: 512 MiB of scores
    for b in range(B):
        for h in range(H):
            kt, vh = k[b, h].double().t().contiguous(), v[b, h].double()
            for r in range(0, S, step):
                s = (q[b, h, r:r + step].double() @ kt) * D ** -0.5
                if case["causal"]:
                    s.masked_fill_(keys[None, :] > keys[r:r + step, None], float("-inf"))
                m = s.amax(dim=-1, keepdim=True)
                s = s.sub_(m).exp_()
                total = s.sum(dim=-1, keepdim=True)
                o[b, h, r:r + step] = (s @ vh) / total
                lse[b, h, r:r + step] = (m + total.log()).squeeze(-1)
    return (o, lse) if case["lse"] else o
