"""The attention calls this repository's speed is judged by.

Each case is one call of a public operator, ``piper_attention`` or ``sage_attention_2pp``, on Q, K
and V resident on the GPU: prep and attention, as a program calls them.  Sizes are the
repository's benchmark workloads (``piper_kernels/workloads.py``), the shapes of its tests, or
generic ones.  ``kind`` is the distribution family of those workloads: "plain" (all standard
normal) or "bias" (a per-channel offset on K and a per-feature offset on V, what trained
projections show and what the operators' smoothing and centring are for).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "piper-kernels_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from piper_kernels import piper_attention, sage_attention_2pp  # noqa: E402

_OPERATORS = {"piper": piper_attention, "sage": sage_attention_2pp}
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, operator, batch, heads, sq, sk, d, dtype, causal=False, kind="plain", layout="bhsd"):
    case = {"operator": operator, "batch": batch, "heads": heads, "sq": sq, "sk": sk, "d": d, "dtype": dtype,
            "causal": causal, "kind": kind, "layout": layout}
    return {"name": name, **case} if name else case


def listed():
    return [
        # the smallest call: short ragged cross-attention, all latency and launches
        _case("piper-tiny-cross", "piper", 1, 4, 35, 67, 64, "fp16"),
        # a short self-attention layer (workload c1)
        _case("piper-short-d64", "piper", 1, 8, 1024, 1024, 64, "fp16", kind="bias"),
        # ragged cross-attention to a short context, as a conditioning layer has it
        _case("piper-ragged-cross", "piper", 2, 12, 1000, 333, 128, "bf16"),
        # a short causal prompt of odd length, batched
        _case("piper-causal-short", "piper", 2, 16, 1531, 1531, 128, "bf16", causal=True),
        # a chunk of queries against a long context, as chunked generation has it
        _case("piper-few-queries", "piper", 1, 24, 256, 16384, 128, "fp16", kind="bias"),
        # a self-attention layer of an image model (workload c2)
        _case("piper-mid", "piper", 1, 24, 4096, 4096, 128, "fp16", kind="bias"),
        # small heads, inputs as the projections leave them: [B, S, H, D] storage seen as [B, H, S, D]
        _case("piper-mid-d64-view", "piper", 2, 20, 4096, 4096, 64, "bf16", layout="bshd"),
        # a long causal prefill (workload c4)
        _case("piper-causal-long", "piper", 4, 32, 8192, 8192, 128, "bf16", causal=True),
        # the headline: a long self-attention layer of a video model (workload c3)
        _case("piper-long", "piper", 1, 24, 16384, 16384, 128, "fp16", kind="bias"),
        # SageAttention2++ at a short layer, an ordinary one and a long causal prefill
        _case("sage-short-d64", "sage", 1, 8, 1024, 1024, 64, "fp16", kind="bias"),
        _case("sage-mid", "sage", 1, 24, 4096, 4096, 128, "fp16", kind="bias"),
        _case("sage-causal-long", "sage", 4, 32, 8192, 8192, 128, "bf16", causal=True),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Lengths over 16 .. 32768 (odd ones among them), both operators, head sizes, dtypes, layouts and
    directions; at most the work and the bytes of the largest listed cases."""
    while True:
        form = rng.choice(("self", "self", "causal", "cross"))
        sq = _log_uniform(rng, 16, 32768)
        sk = _log_uniform(rng, 16, 32768) if form == "cross" else sq
        if rng.random() < 0.4:  # whole tiles are the most frequent lengths in use
            sq, sk = max(64, sq // 64 * 64), max(64, sk // 64 * 64)
        case = _case(None, rng.choice(("piper", "piper", "sage")), rng.choice((1, 1, 2, 4)), _log_uniform(rng, 1, 40), sq, sk,
                     rng.choice((64, 128)), rng.choice(("fp16", "bf16")), causal=form == "causal",
                     kind=rng.choice(("plain", "bias")), layout=rng.choice(("bhsd", "bhsd", "bshd")))
        cost = work(case)
        if cost["flops"] <= 3.3e12 and cost["bytes"] <= 1.1e9:
            return case


def _tensors(case, seed):
    b, h, sq, sk, d = (case[k] for k in ("batch", "heads", "sq", "sk", "d"))
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    def made(length, offset=0.0):
        x = normal(b, h, length, d)
        if offset:
            x += offset * normal(b, h, 1, d)
        x = x.to(dtype)
        # the same values; "bshd" keeps each token's heads together in memory
        return x if case["layout"] == "bhsd" else x.transpose(1, 2).contiguous().transpose(1, 2)

    bias = case["kind"] == "bias"
    return made(sq), made(sk, math.sqrt(2.0) if bias else 0.0), made(sk, 2.0 if bias else 0.0)


def prepare(case, seed):
    return {"operator": _OPERATORS[case["operator"]], "qkv": _tensors(case, seed), "causal": case["causal"]}


def run(state):
    q, k, v = state["qkv"]
    return state["operator"](q, k, v, is_causal=state["causal"])


def work(case):
    b, h, sq, sk, d = (case[k] for k in ("batch", "heads", "sq", "sk", "d"))
    pairs = sq * (sq + 1) // 2 if case["causal"] else sq * sk
    return {"bytes": 2 * b * h * d * (2 * sq + 2 * sk), "flops": 4 * b * h * d * pairs}


def tolerance(case):
    """About four times what summing the 64-key blocks in another order changes (K and V permuted by
    blocks: every P code's block stays whole, the K mean and the sums round differently).

    Piper Attention: 1.8e-5 relative in fp16 and 6.8e-5 in bf16, single values by one ulp of the
    output (9.8e-4, 7.8e-3) or by one UINT8 code of P.  SageAttention2++ rounds P to FP8 relative to a
    running maximum, so the order changes the codes themselves: 3e-3 relative with biased V, 3.6e-2
    (bounded here by 3e-2) with zero-mean V, where the output is all cancellation."""
    if case["operator"] == "sage":
        return {"rel": 0.012, "max": 0.06} if case["kind"] == "bias" else {"rel": 0.03, "max": 0.95}
    return {"rel": 1e-4, "max": 0.02} if case["dtype"] == "fp16" else {"rel": 4e-4, "max": 0.05}


def exact(case, seed):
    """Softmax attention of the same inputs in FP64, head by head: the operators' 8-bit codes are part
    of their distance from it (about 2%)."""
    q, k, v = _tensors(case, seed)
    b, h, sq, sk, d = (case[x] for x in ("batch", "heads", "sq", "sk", "d"))
    out = torch.empty((b, h, sq, d), device="cuda", dtype=torch.float64)
    rows = max(1, (1 << 25) // sk)  # query rows at a time: 256 MiB of scores
    for i in range(b):
        for j in range(h):
            kt, vd = k[i, j].double().t().contiguous(), v[i, j].double()
            for r in range(0, sq, rows):
                s = torch.mm(q[i, j, r : r + rows].double() * d**-0.5, kt)
                if case["causal"]:
                    s.masked_fill_(torch.arange(sk, device="cuda")[None] > torch.arange(r, r + s.shape[0], device="cuda")[:, None],
                                   -math.inf)
                s.sub_(s.amax(dim=1, keepdim=True)).exp_()
                total = s.sum(dim=1, keepdim=True)
                out[i, j, r : r + rows] = torch.mm(s, vd) / total
    return out
