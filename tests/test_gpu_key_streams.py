"""Key streams (csrc/attention.hip attention_streams_kernel): two and four parts of small grids, at the
edges -- fewer key tiles than streams, key tiles that do not divide, query rows past the end in one of a
workgroup's groups, one row -- against the unsplit kernel and the oracle; the two-step and the fused
entry points bit for bit alike.  The balanced entry points, which choose streams themselves (causal Piper
Attention, SageAttention2++), bit for bit the others, scores whose block maxima grow, leave the
subtraction-free range or are not finite among them; a batch-head's output bit for bit the same alone and
in a batch."""

from __future__ import annotations

import pytest
import torch

from _parity import assert_attention_close, gpu_attention, gpu_prepare, log, oracle_attention
from oracle import piper_oracle as oracle
from piper_kernels._hip import library as native
from piper_kernels.attention.piper_attention._plan import MI355XPlan

pytestmark = pytest.mark.gpu

SHAPES = [
    # (B, H, Sq, Sk)
    (1, 1, 1, 1),  # one key tile: three of four streams see no key
    (1, 2, 33, 65),
    (2, 3, 97, 700),  # 11 key tiles, the last 60 keys
    (1, 4, 130, 1024),
]


@pytest.mark.parametrize("granularity", ["per_thread", "per_warp"])
@pytest.mark.parametrize("parts", [2, 4])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_streams_match_the_unsplit_kernel_and_the_oracle(shape, d, parts, granularity, gfx950_device) -> None:
    b, h, sq, sk = shape
    log(f"[case] key streams {shape} D={d} parts={parts} {granularity}")
    g = torch.Generator().manual_seed(sq + sk + d)
    q = torch.randn((b, h, sq, d), generator=g).to(torch.float16)
    k, v = ((torch.randn((b, h, sk, d), generator=g) + torch.randn((b, h, 1, d), generator=g)).to(torch.float16)
            for _ in range(2))
    plans = [MI355XPlan(waves=4, three_per_cu=True, key_parts=p) for p in (1, parts)]
    whole, split = (gpu_attention(gpu_prepare(q, k, v, d**-0.5, False, gfx950_device, plan=p, quantize_query=False,
                                              qk_granularity=granularity), torch.float32) for p in plans)
    two_step = gpu_prepare(q, k, v, d**-0.5, False, gfx950_device, plan=plans[1], qk_granularity=granularity)
    assert torch.equal(gpu_attention(two_step, torch.float32), split)
    assert torch.equal(gpu_attention(two_step, torch.float16), split.to(torch.float16))
    # the streams' FP32 sums enter in another order: a few ulps of a value of the outputs' size
    assert (split - whole).abs().max().item() <= 1e-5 * max(1.0, whole.abs().max().item())
    expected, bound = oracle_attention(oracle.prepare(q, k, v, False, granularity), d**-0.5, False)
    assert_attention_close(split.cpu().numpy(), expected, f"{parts} streams", flip_bound=bound)


class _Balanced:
    """The library with its attention entry points replaced by the balanced ones."""

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        return getattr(self._lib, {"attention_forward_fused": "attention_forward_balanced",
                                   "sage_attention_forward": "sage_attention_forward_balanced"}.get(name, name))


BALANCED = [
    # (operator, B, H, Sq, Sk, causal): four streams, two streams, a grid past the rule's lines
    ("piper", 1, 3, 500, 500, True),
    ("piper", 1, 12, 1031, 1031, True),
    ("piper", 2, 30, 1031, 1031, True),
    ("sage", 1, 3, 500, 500, True),
    ("sage", 1, 12, 1031, 1031, True),
    ("sage", 1, 5, 97, 300, False),
    ("sage", 1, 40, 257, 700, False),
    ("sage", 2, 40, 257, 700, False),
    ("sage", 1, 2, 100, 8257, False),  # more than 128 key tiles
    ("sage", 1, 1, 4500, 4500, True),
]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", BALANCED, ids=str)
def test_balanced_entry_points_equal_the_others_bit_for_bit(case, d, gfx950_device, monkeypatch) -> None:
    from piper_kernels.attention.piper_attention.hip import _launch_piper_attention, _prepare_piper_attention
    from piper_kernels.attention.sage_attention_2pp.hip import _launch_sage_attention_2pp, _prepare_sage_attention_2pp

    operator, b, h, sq, sk, causal = case
    log(f"[case] balanced {case} D={d}")
    g = torch.Generator().manual_seed(sq + h)
    q = torch.randn((b, h, sq, d), generator=g).to(torch.bfloat16).to(gfx950_device)
    k, v = (torch.randn((b, h, sk, d), generator=g).to(torch.bfloat16).to(gfx950_device) for _ in range(2))
    lib = native.load_library()
    outs = []
    for handle in (lib, _Balanced(lib)):
        monkeypatch.setattr(native, "load_library", lambda *a, handle=handle: handle)
        out = torch.empty((b, h, sq, d), device=gfx950_device)
        if operator == "piper":
            prepared = _prepare_piper_attention(q, k, v, d**-0.5, causal, quantize_query=False)
            outs.append(_launch_piper_attention(prepared, output=out))
        else:
            outs.append(_launch_sage_attention_2pp(_prepare_sage_attention_2pp(q, k, v, d**-0.5, causal), output=out))
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("granularity", ["per_thread", "per_warp"])
@pytest.mark.parametrize("operator", ["piper", "sage"])
@pytest.mark.parametrize("d", [64, 128])
def test_growing_and_extreme_scores_bit_for_bit(d, operator, granularity, gfx950_device, monkeypatch) -> None:
    """Keys that grow along the sequence (the frame moves in most tiles), rows of large queries (block maxima past
    the subtraction-free range), an infinite and a NaN value: two and four streams against the other kernels."""
    from piper_kernels.attention.sage_attention_2pp.hip import _launch_sage_attention_2pp, _prepare_sage_attention_2pp

    log(f"[case] streams, extreme scores {operator} D={d} {granularity}")
    g = torch.Generator().manual_seed(d)
    lib = native.load_library()
    for heads, causal, bad in ((2, False, False), (2, True, False), (9, True, False), (2, False, True), (2, True, True)):
        if operator == "piper" and not causal:
            continue
        s = 1000
        q = torch.randn((1, heads, s, d), generator=g)
        q[:, :, 100:200] *= 60
        k = torch.randn((1, heads, s, d), generator=g) * torch.linspace(0.1, 12, s).reshape(1, 1, s, 1)
        v = torch.randn((1, heads, s, d), generator=g)
        v[:, :, 37] *= 1000
        if bad:
            q[:, 0, 5, 3], v[:, 0, 300, 2], k[:, 1, 700, 1] = float("nan"), float("inf"), float("inf")
        q, k, v = (x.to(torch.bfloat16).to(gfx950_device) for x in (q, k, v))
        outs = []
        for handle in (lib, _Balanced(lib)):
            monkeypatch.setattr(native, "load_library", lambda *a, handle=handle: handle)
            if operator == "sage":
                out = torch.empty((1, heads, s, d), device=gfx950_device)
                p = _prepare_sage_attention_2pp(q, k, v, d**-0.5, causal, qk_granularity=granularity)
                outs.append(_launch_sage_attention_2pp(p, output=out))
            else:
                outs.append(gpu_attention(gpu_prepare(q, k, v, d**-0.5, causal, gfx950_device, quantize_query=False,
                                                      qk_granularity=granularity)))
        assert torch.allclose(outs[0], outs[1], rtol=0, atol=0, equal_nan=True)
        assert bad or torch.isfinite(outs[0]).all()


@pytest.mark.parametrize("operator", ["piper", "sage"])
@pytest.mark.parametrize("d", [64, 128])
def test_a_batch_head_alone_and_in_a_batch(d, operator, gfx950_device) -> None:
    """The public operators choose streams by the grid: four, two or none for one, six and many batch-heads."""
    from piper_kernels import piper_attention, sage_attention_2pp

    public = piper_attention if operator == "piper" else sage_attention_2pp
    log(f"[case] batch against alone {operator} D={d}")
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn((2, 40, 1031, d), generator=g).to(torch.float16).to(gfx950_device) for _ in range(3))
    with torch.no_grad():
        for causal in (True,) if operator == "piper" else (True, False):
            want = public(q, k, v, is_causal=causal)
            for heads in (1, 6, 14):
                got = public(q[1:, :heads], k[1:, :heads], v[1:, :heads], is_causal=causal)
                assert torch.equal(got, want[1:, :heads]), heads
