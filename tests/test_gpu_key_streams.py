"""Key streams (csrc/attention.hip attention_streams_kernel): two and four parts of small grids, at the
edges -- fewer key tiles than streams, key tiles that do not divide, query rows past the end in one of a
workgroup's groups, one row -- against the unsplit kernel and the oracle; the two-step and the fused
entry points bit for bit alike.  The balanced entry points, which choose streams themselves (causal Piper
Attention, SageAttention2++), against the others."""

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
]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", BALANCED, ids=str)
def test_balanced_entry_points_equal_the_others_to_rounding(case, d, gfx950_device, monkeypatch) -> None:
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
    # every probability code is the same (an FP8 code off by one step would show as 1e-3); the FP32 sums
    # enter in another order: a few ulps of a value of the outputs' size
    assert (outs[0] - outs[1]).abs().max().item() <= 2e-6 * max(1.0, outs[0].abs().max().item())
