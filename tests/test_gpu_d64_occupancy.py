"""Head size 64 with four 4-wave workgroups per CU (csrc/kernels.h waves_per_simd): grids just over
and just under one round of 1024 workgroups, under hardware dispatch and from the work queue's
persistent grid, against the two-waves-per-SIMD plan bit for bit."""

from __future__ import annotations

import pytest
import torch

from _parity import gpu_attention, gpu_prepare, log
from piper_kernels.attention.piper_attention._plan import MI355XPlan

pytestmark = pytest.mark.gpu

CASES = [
    # (B, H, S, causal): query tiles of 128 rows
    (1, 18, 7297, False),  # 18 x 58 = 1044 tiles: over one round, the last tile of a head one row
    (1, 18, 7297, True),
    (3, 17, 2560, True),  # 51 x 20 = 1020 tiles: under one round
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}-{'causal' if c[3] else 'full'}")
def test_four_workgroups_per_cu_match_the_two_wave_plan(case, gfx950_device) -> None:
    b, h, s, causal = case
    log(f"[case] D = 64 occupancy {case}")
    g = torch.Generator().manual_seed(s + h)
    q, k, v = (torch.randn((b, h, s, 64), generator=g).to(torch.float16) for _ in range(3))
    outs = []
    for plan in (MI355XPlan(waves=8), MI355XPlan(waves=4, three_per_cu=True),
                 MI355XPlan(waves=4, three_per_cu=True, work_queue=True)):
        prepared = gpu_prepare(q, k, v, 0.125, causal, gfx950_device, plan=plan, quantize_query=False)
        outs.append(gpu_attention(prepared, torch.float32))
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])
