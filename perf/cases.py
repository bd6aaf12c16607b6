"""The calls whose speed matters to a user of this package, for timing and comparing builds.

A case names a call of the public entry points (`fa.forward`, `fa.forward_lse`,
`fa.forward_splitkv`) by its shape [batch, heads, seqlen, head_dim], mask, options and input
distribution. `listed()` holds fixed cases from the smallest launch to the largest, `draw()` one
more of the same ranges, `prepare()` the inputs on the GPU, `run()` one call, `exact()` its result
in 64 bits from plain torch.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "flash-attention-from-scratch_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import fa  # noqa: E402


def _case(name, op, batch, heads, seqlen, head_dim, causal, std=1.0, boost=1.0):
    return {"name": name, "op": op, "batch": batch, "heads": heads, "seqlen": seqlen,
            "head_dim": head_dim, "causal": causal, "std": std, "boost": boost}


def listed():
    return [
        # A single short sequence through a small model: one launch, nothing but latency.
        _case("tiny_d64", "forward", 1, 4, 256, 64, False),
        # Two prompts of odd length through a small decoder: a grid that leaves most CUs idle.
        _case("small_ragged_d64_causal", "forward", 2, 8, 1000, 64, True),
        # Prefill of one prompt, 16 heads of 128: the commonest serving call.
        _case("prompt_d128_causal", "forward", 1, 16, 2000, 128, True),
        # A batch of short sequences in training or batched prefill.
        _case("short_batch_d128_causal", "forward", 32, 16, 512, 128, True),
        # A bidirectional encoder over a batch of texts or images, ragged length.
        _case("encoder_ragged_d64", "forward", 16, 32, 1000, 64, False),
        # A decoder batch with many heads of 64 whose keys have a few large outliers.
        _case("many_heads_d64_causal", "forward", 16, 32, 2048, 64, True, std=0.5, boost=8.0),
        # Training at 4k context, heads of 128.
        _case("train_4k_d128_causal", "forward", 4, 16, 4096, 128, True),
        # The forward of a training step that keeps the row log-sum-exp for its backward, or one
        # hop of context parallelism; bidirectional, ragged.
        _case("lse_ragged_d128", "lse", 4, 16, 3001, 128, False),
        # One GPU's share of a long prompt under tensor parallelism: two heads of 16k keys.
        _case("few_heads_16k_d128_causal", "forward", 1, 2, 16384, 128, True),
        # The same with heads of 64, bidirectional, asking for split-KV by name.
        _case("splitkv_8k_d64", "splitkv", 1, 4, 8192, 64, False),
        # Long context, both masks: the largest calls.
        _case("long_16k_d128", "forward", 1, 16, 16384, 128, False),
        _case("long_16k_d128_causal", "forward", 1, 16, 16384, 128, True),
    ]


# The largest listed call: 4 * 16 heads * 16384^2 * 128 FLOPs.
_MOST_FLOPS = 4.0 * 16 * 16384**2 * 128


def draw(rng):
    op = rng.choice(["forward"] * 6 + ["lse", "splitkv"])
    head_dim = rng.choice([64, 128])
    causal = rng.random() < 0.5
    seqlen = int(round(math.exp(rng.uniform(math.log(64), math.log(16384)))))
    if rng.random() < 0.4:  # lengths that programs pad to
        seqlen = max(64, seqlen // 64 * 64)
    heads = rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 20, 24, 32, 40])
    batch = int(round(math.exp(rng.uniform(0, math.log(32)))))
    while 4.0 * batch * heads * seqlen**2 * head_dim > _MOST_FLOPS:
        if batch > 1:
            batch //= 2
        else:
            heads = (heads + 1) // 2
    case = _case("", op, batch, heads, seqlen, head_dim, causal,
                 std=rng.choice([0.5, 1.0, 1.0]), boost=rng.choice([1.0, 1.0, 1.0, 8.0]))
    del case["name"]
    return case


def prepare(case, seed):
    """q, k, v fp16 ~ N(0, std^2); with `boost`, 1 % of each head's key rows times `boost` (the
    outlier keys of trained models)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["batch"], case["heads"], case["seqlen"], case["head_dim"])
    q, k, v = (torch.randn(shape, generator=g, device="cuda").mul_(case["std"])
               for _ in range(3))
    outliers = case["seqlen"] // 100
    if case["boost"] != 1.0 and outliers:
        rows = torch.rand(shape[:3], generator=g, device="cuda").topk(outliers).indices
        scale = torch.ones(shape[:3], device="cuda").scatter_(2, rows, case["boost"])
        k.mul_(scale.unsqueeze(3))
    return {"op": case["op"], "causal": case["causal"], "q": q.half(), "k": k.half(),
            "v": v.half()}


def run(state):
    q, k, v, causal = state["q"], state["k"], state["v"], state["causal"]
    if state["op"] == "lse":
        return fa.forward_lse(q, k, v, causal=causal)
    if state["op"] == "splitkv":
        return fa.forward_splitkv(q, k, v, causal=causal)
    return fa.forward(q, k, v, causal=causal)


def work(case):
    """Q, K, V read once, O (and the LSE) written once; two products over the visible (query,
    key) pairs."""
    rows = case["batch"] * case["heads"] * case["seqlen"]
    keys = (case["seqlen"] + 1) / 2 if case["causal"] else case["seqlen"]
    lse = 0 if case["op"] == "forward" else 4 * rows
    return {"bytes": 4 * rows * case["head_dim"] * 2 + lse,
            "flops": 4.0 * rows * keys * case["head_dim"]}


def tolerance(case):
    # fp16 output and fp16 probabilities, each rounded by up to 2^-11. Two of the package's own
    # kernels (the simple "baseline" tile and the default) differ by at most 4e-4 (2-norm) and
    # 1e-2 (one value: a sum of cancelling terms in a causal row of few keys) over these ranges;
    # either is within 3e-4 of 64 bits. Four times that.
    return {"rel": 1.5e-3, "max": 4e-2}


def exact(case, seed):
    state = prepare(case, seed)
    q, k, v = (state[x].flatten(0, 1) for x in "qkv")
    heads, n, d = q.shape
    out = torch.empty(heads, n, d, dtype=torch.float64, device=q.device)
    lse = torch.empty(heads, n, dtype=torch.float64, device=q.device)
    cols = torch.arange(n, device=q.device)
    rows = max(1, min(n, 2**27 // n))          # about 1 GiB of scores at a time
    group = max(1, 2**27 // (n * rows))
    for h in range(0, heads, group):
        qh, kh, vh = (x[h:h + group].double() for x in (q, k, v))
        kt = kh.transpose(1, 2).contiguous()
        for i in range(0, n, rows):
            s = torch.matmul(qh[:, i:i + rows].contiguous(), kt) / math.sqrt(d)
            if case["causal"]:
                s.masked_fill_(cols > cols[i:i + rows, None], -math.inf)
            lse[h:h + group, i:i + rows] = torch.logsumexp(s, dim=2)
            s = torch.exp(s - lse[h:h + group, i:i + rows, None])
            out[h:h + group, i:i + rows] = torch.matmul(s, vh)
    shape = (case["batch"], case["heads"], n)
    out = out.view(*shape, d)
    return out if case["op"] == "forward" else (out, lse.view(shape))
