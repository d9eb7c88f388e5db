"""The single-pass prep's bounded-wait fallback on MI355X, forced from the host.

A chunk of the single pass waits for its batch-head tensor's mean, which the tensor's last chunk
publishes; the wait is bounded, and a chunk whose wait ends computes the mean itself from K/V in
HBM in the same cascade order (csrc/prep.hip, column_mean_from_rows) and is counted in the prep's
status word.  PIPER_PREPARE_SELF_MEAN makes every waiting chunk take that path at once (a wait of
zero polls), so every kernel still runs to its normal end: the codes, scales and means must be
bit-identical to the ordinary prep (and to the oracle, the reference's torch.mean order), and the
status word must count exactly the chunks that waited: (chunks - 1) per centred tensor.  The ordinary
prep of up to 32 chunks takes another route (short or two-pass), of more the single pass itself.
SageAttention2++'s V chunks wait for their channel scales (column_scale_from_rows); its prep counts
nothing, so its forced path is checked by its bytes alone.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _parity import assert_prep_bit_exact, log, prepared_numpy
from oracle import piper_oracle as oracle
from piper_kernels._hip import library as native

pytestmark = pytest.mark.gpu

CASES = [
    # (B, H, Sq, Sk, dtype, causal)
    (1, 3, 4096, 4096, torch.float16, False),  # 16 chunks
    (2, 2, 1000, 1000, torch.bfloat16, False),  # 4 chunks, the last short (ragged)
    (1, 2, 16384, 16384, torch.float16, False),  # 64 chunks
    (1, 1, 32768, 32768, torch.float16, False),  # 128 chunks: the single pass's longest sequence
    (1, 2, 4096, 4096, torch.bfloat16, True),  # causal: only K is centred and waits
    (1, 1, 100, 100, torch.float16, False),  # one chunk: it is its tensor's last, nothing waits
    (1, 2, 300, 8450, torch.bfloat16, False),  # 34 chunks, the last ragged: the ordinary prep waits too
    (2, 1, 8300, 8300, torch.float16, True),
]


def _inputs(case, seed, d=128):
    b, h, sq, sk, dtype, _ = case
    g = torch.Generator().manual_seed(seed)
    q = torch.randn((b, h, sq, d), generator=g).to(dtype)
    k = (torch.randn((b, h, sk, d), generator=g) + 2 * torch.randn((b, h, 1, d), generator=g)).to(dtype)
    v = (torch.randn((b, h, sk, d), generator=g) + 4 * torch.randn((b, h, 1, d), generator=g)).to(dtype)
    return q, k, v


def _prepare(q, k, v, causal, device, flags, static=False):
    from piper_kernels.attention.piper_attention.hip import _prepare_piper_attention

    b, h, sq, d = q.shape
    shape = native.PiperShape(b, h, sq, k.shape[2], d)
    lib = native.load_library()
    workspace = None
    if not static:
        workspace = torch.empty(lib.prepared_layout(shape).workspace_bytes, dtype=torch.uint8, device=device)
    with torch.no_grad():
        # the two-step prep: the single pass's grid also carries the query blocks
        prepared = _prepare_piper_attention(q.to(device), k.to(device), v.to(device), d**-0.5, causal,
                                            workspace=workspace, static_workspace=static, prep_flags=flags)
    stream = torch.cuda.current_stream(device)
    status = lib.prepare_status(shape, None if static else workspace.data_ptr(), stream.cuda_stream)
    return prepared, status


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}x{c[3]}-{str(c[4])[6:]}-{'causal' if c[5] else 'full'}")
def test_self_computed_means_are_bit_identical_and_counted(case, d, gfx950_device) -> None:
    b, h, sq, sk, dtype, causal = case
    chunks = -(-sk // 256)
    log(f"[case] prep fallback {case} D={d}: {chunks} chunks per tensor")
    q, k, v = _inputs(case, 4100 + sq, d)
    normal, normal_status = _prepare(q, k, v, causal, gfx950_device, 0)
    forced, forced_status = _prepare(q, k, v, causal, gfx950_device, native.PREPARE_SELF_MEAN)
    centred = 1 if causal else 2
    expected_count = (chunks - 1) * centred * b * h
    log(f"  status: ordinary {normal_status}, forced {forced_status} (expected {expected_count})")
    assert normal_status == 0
    assert forced_status == expected_count
    got, want = prepared_numpy(forced), prepared_numpy(normal)
    for name, value in want.items():
        if value is None:
            assert got[name] is None, name
            continue
        assert np.array_equal(np.ascontiguousarray(got[name]).view(np.uint8),
                              np.ascontiguousarray(value).view(np.uint8)), f"{name} differs on the fallback path"
    if sk <= 4096:  # the oracle: the reference's torch.mean order and codes
        assert_prep_bit_exact(got, oracle.prepare(q, k, v, causal, "per_thread"), forced.shape, causal)


def test_static_scratch_status_counts_the_forced_fallback(gfx950_device) -> None:
    case = (1, 2, 300, 8400, torch.float16, False)  # 33 chunks: the ordinary prep is the single pass too
    log(f"[case] piper_prepare_static fallback {case}")
    q, k, v = _inputs(case, 77)
    forced, status = _prepare(q, k, v, False, gfx950_device, native.PREPARE_SELF_MEAN, static=True)
    assert status == (33 - 1) * 2 * 2
    normal, status = _prepare(q, k, v, False, gfx950_device, 0, static=True)
    assert status == 0  # each call clears the word it counts in
    got, want = prepared_numpy(forced), prepared_numpy(normal)  # every byte the header specifies
    for name, value in want.items():
        assert np.array_equal(np.ascontiguousarray(got[name]).view(np.uint8),
                              np.ascontiguousarray(value).view(np.uint8)), f"{name} differs on the fallback path"


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("case", [c for c in CASES if not c[5]], ids=lambda c: f"{c[0]}x{c[1]}x{c[3]}-{str(c[4])[6:]}")
def test_sage_self_computed_statistics_are_bit_identical(case, d, gfx950_device) -> None:
    from oracle import sage2pp_oracle
    from piper_kernels.attention.sage_attention_2pp.hip import _prepare_sage_attention_2pp

    _, _, sq, sk, _, _ = case
    log(f"[case] sage prep fallback {case} D={d}")
    q, k, v = _inputs(case, 5200 + sk, d)
    got = []
    for flags in (0, native.PREPARE_SELF_MEAN):
        with torch.no_grad():
            p = _prepare_sage_attention_2pp(*(x.to(gfx950_device) for x in (q, k, v)), d**-0.5, False, prep_flags=flags)
        torch.cuda.synchronize(gfx950_device)
        got.append({"key_code": p.key_code().cpu().numpy(), "value_code": p.value_code().cpu().numpy(),
                    "key_scale": p.key_scale.cpu().numpy(), "key_mean": p.key_mean.cpu().numpy(),
                    "value_scale": p.value_scale.cpu().numpy()})
    for name, value in got[0].items():
        assert np.array_equal(value.view(np.uint8), got[1][name].view(np.uint8)), f"{name} differs on the fallback path"
    if sk <= 8450:
        want = sage2pp_oracle.prepare(q, k, v, "per_thread")
        assert np.array_equal(got[1]["value_code"][:, :, :sk], want["value_code"])
        assert np.array_equal(got[1]["key_code"][:, :, :sk], want["key_code"])
        for name in ("key_mean", "value_scale"):
            assert np.array_equal(got[1][name].reshape(-1).view(np.uint32),
                                  np.ascontiguousarray(want[name], dtype=np.float32).reshape(-1).view(np.uint32)), name
