"""Causal grids dispatched longest first across heads (csrc/stream.h workgroup_tile): every tile is
computed once whatever the order, so the output equals the forward order's bit for bit -- with
batch-heads that divide over the 8 XCDs, that do not, and fewer than 8, for both operators."""

from __future__ import annotations

import pytest
import torch

from _parity import gpu_attention, gpu_prepare, log
from piper_kernels.attention.piper_attention._plan import MI355XPlan

pytestmark = pytest.mark.gpu

ORDERS = [MI355XPlan(waves=4, three_per_cu=True, causal_longest_first=f, xcd_remap=x, causal_interleave=i)
          for f, x, i in ((False, True, False), (True, True, False), (True, True, True), (True, False, False))]


@pytest.mark.parametrize("operator", ["piper", "sage"])
@pytest.mark.parametrize("shape", [(2, 8, 700, 128), (3, 5, 451, 128), (1, 3, 1000, 64), (1, 1, 64, 64)], ids=str)
def test_every_tile_order_is_bit_identical(shape, operator, gfx950_device) -> None:
    from piper_kernels.attention.sage_attention_2pp.hip import _launch_sage_attention_2pp, _prepare_sage_attention_2pp

    b, h, s, d = shape
    log(f"[case] tile order {operator} {shape}")
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn((b, h, s, d), generator=g).to(torch.bfloat16) for _ in range(3))
    outs = []
    for plan in ORDERS:
        if operator == "piper":
            outs.append(gpu_attention(gpu_prepare(q, k, v, d**-0.5, True, gfx950_device, plan=plan), torch.float32))
        else:
            with torch.no_grad():
                prepared = _prepare_sage_attention_2pp(q.to(gfx950_device), k.to(gfx950_device), v.to(gfx950_device),
                                                       d**-0.5, True, plan=plan)
                outs.append(_launch_sage_attention_2pp(prepared, output=torch.empty((b, h, s, d), device=gfx950_device)))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
