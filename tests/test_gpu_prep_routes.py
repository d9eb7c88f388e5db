"""The prep's routes (csrc/prep.hip launch_prep_typed) agree bit for bit: a batch-head's codes, scales
and statistics do not depend on how many other batch-heads the call has, while the route does (short,
two-pass, single pass).  Lengths at the edges of 16-row blocks, 64-row units and 256-row chunks, and just
beyond the single pass's longest (the statistics' own kernel), against the oracle, on strided inputs."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _parity import assert_prep_bit_exact, gpu_prepare, log, prepared_numpy
from oracle import piper_oracle as oracle
from oracle import sage2pp_oracle

pytestmark = pytest.mark.gpu

ROUTES = [
    # (D, S, few heads, many heads): short against single pass, two-pass against single pass (D = 128);
    # short against two-pass, two-pass against single pass (D = 64)
    (128, 1000, 2, 68),
    (128, 5003, 2, 16),
    (64, 1000, 2, 68),
    (64, 8100, 1, 66),
]


def _inputs(b, h, s, d, seed):
    g = torch.Generator().manual_seed(seed)
    # [B, S, H, D] storage: rows of a head are strided
    q, k, v = (torch.randn((b, s, h, d), generator=g) for _ in range(3))
    return tuple(x.to(torch.bfloat16).transpose(1, 2) for x in (q, k + 1.5, v - 2.0))


def _sage(q, k, v, causal, device):
    from piper_kernels.attention.sage_attention_2pp.hip import _prepare_sage_attention_2pp

    with torch.no_grad():
        p = _prepare_sage_attention_2pp(q.to(device), k.to(device), v.to(device), q.shape[-1] ** -0.5, causal)
    torch.cuda.synchronize(device)
    return {"key_code": p.key_code().cpu().numpy(), "value_code": p.value_code().cpu().numpy(),
            "key_scale": p.key_scale.cpu().numpy(), "key_mean": p.key_mean.cpu().numpy(),
            "value_scale": p.value_scale.cpu().numpy()}


@pytest.mark.parametrize("operator,causal", [("piper", False), ("piper", True), ("sage", False)])
@pytest.mark.parametrize("route", ROUTES, ids=str)
def test_routes_agree_bit_for_bit(route, operator, causal, gfx950_device) -> None:
    d, s, few, many = route
    log(f"[case] prep routes {operator} {route} causal={causal}")
    q, k, v = _inputs(1, many, s, d, s + d)
    run = _sage if operator == "sage" else (
        lambda *a: prepared_numpy(gpu_prepare(*a[:3], d**-0.5, a[3], a[4], qk_granularity="per_thread")))
    big = run(q, k, v, causal, gfx950_device)
    small = run(q[:, :few], k[:, :few], v[:, :few], causal, gfx950_device)
    for name, value in small.items():
        got = np.ascontiguousarray(big[name][:, :few]).view(np.uint8)
        assert np.array_equal(np.ascontiguousarray(value).view(np.uint8), got), f"{name} differs"


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s", [1, 15, 16, 17, 64, 255, 256, 257, 1023, 1024, 1025, 1300])
def test_edge_lengths_match_the_oracle(s, d, gfx950_device) -> None:
    _check_against_the_oracle(s, d, 2, gfx950_device)


@pytest.mark.parametrize("d", [64, 128])
def test_past_the_single_pass_matches_the_oracle(d, gfx950_device) -> None:
    _check_against_the_oracle(32768 + 257, d, 1, gfx950_device)


def _check_against_the_oracle(s, d, heads, gfx950_device) -> None:
    log(f"[case] prep length {s} D={d}")
    q, k, v = _inputs(1, heads, s, d, 7 * s + d)
    for causal in (False, True):
        prepared = gpu_prepare(q, k, v, d**-0.5, causal, gfx950_device, qk_granularity="per_thread")
        assert_prep_bit_exact(prepared_numpy(prepared), oracle.prepare(q, k, v, causal, "per_thread"), prepared.shape, causal)
    got, want = _sage(q, k, v, False, gfx950_device), sage2pp_oracle.prepare(q, k, v, "per_thread")
    assert np.array_equal(got["value_code"][:, :, :s], want["value_code"]) and not got["value_code"][:, :, s:].any()
    assert np.array_equal(got["key_code"][:, :, :s], want["key_code"]) and not got["key_code"][:, :, s:].any()
    for name in ("key_mean", "value_scale"):
        assert np.array_equal(got[name].reshape(-1).view(np.uint32),
                              np.ascontiguousarray(want[name], dtype=np.float32).reshape(-1).view(np.uint32)), name
