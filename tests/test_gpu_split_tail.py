"""The key-range split of the query tiles beyond whole rounds of resident workgroups
(csrc/attention.hip attention_w3_kernel, kSplit): the whole tiles' rows equal the unsplit kernel bit
for bit, the split tiles' rows to rounding -- a remainder of a few tiles, one that starts inside a
head, ragged query and key lengths, and more parts than key tiles."""

from __future__ import annotations

import pytest
import torch

from _parity import gpu_attention, gpu_prepare, log
from piper_kernels.attention.piper_attention._plan import MAX_KEY_PARTS, MI355XPlan, split_parts

CASES = [
    # (H, query tiles per head at 256 CUs' slots plus the rest, last tile's rows, Sk, D, parts)
    (7, 110, 128, 257, 128, 3),  # 770 tiles: two beyond the 768 slots
    (5, 171, 35, 300, 128, 2),  # 855 tiles: the remainder starts inside the fifth head
    (9, 116, 1, 700, 64, 8),  # 1044 tiles over 1024 slots at D = 64
    (3, 2, 77, 130, 64, 8),  # fewer tiles than slots, fewer key tiles than parts
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_only_the_last_round_is_split(case, gfx950_device) -> None:
    h, tiles, last, sk, d, parts = case
    sq = (tiles - 1) * 128 + last
    log(f"[case] split tail {case}")
    g = torch.Generator().manual_seed(sq)
    q = torch.randn((1, h, sq, d), generator=g).to(torch.float16)
    k, v = (torch.randn((1, h, sk, d), generator=g).to(torch.float16) for _ in range(2))
    outs = [gpu_attention(gpu_prepare(q, k, v, d**-0.5, False, gfx950_device, quantize_query=False,
                                      plan=MI355XPlan(waves=4, three_per_cu=True, key_parts=p)), torch.float32)
            for p in (1, parts)]
    whole, split = (o.reshape(h * sq, d) for o in outs)
    slots = torch.cuda.get_device_properties(gfx950_device).multi_processor_count * (4 if d == 64 else 3)
    first = h * tiles // slots * slots
    row0 = first // tiles * sq + first % tiles * 128
    assert torch.equal(split[:row0], whole[:row0])
    # the parts' FP32 sums enter in another order: a few ulps of a value of the outputs' size
    assert (split[row0:] - whole[row0:]).abs().max().item() <= 1e-5 * max(1.0, whole.abs().max().item())


def test_the_rule_splits_only_partial_rounds_into_whole_key_tiles() -> None:
    for batch, heads, sq, sk, d in [(1, 24, 256, 16384, 128), (2, 20, 4096, 4096, 64), (1, 28, 5000, 5000, 128),
                                    (1, 1, 1, 1, 64), (1, 3, 129, 64, 128), (4, 40, 32768, 17, 64)]:
        parts = split_parts(batch, heads, sq, sk, d)
        assert 1 <= parts <= MAX_KEY_PARTS and (parts == 1 or 2 * parts <= -(-sk // 64))
    for d, tiles in ((128, 768), (128, 1536), (64, 1024)):  # whole rounds
        assert split_parts(1, 1, 128 * tiles, 4096, d) == 1
    assert split_parts(1, 24, 256, 16384, 128) == 8
    # 192 query tiles still fit the GPU as two key streams each; 320 do not, and six key tiles are too few
    # for partial sums
    assert split_parts(2, 12, 1000, 333, 128) == 2 and split_parts(1, 40, 1000, 333, 128) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_the_split_stays_inside_the_workspace_it_asks_for(case, gfx950_device, monkeypatch) -> None:
    """The bytes piper_attention_workspace_bytes reports on this device: the split rows' partial sums only;
    nothing behind them is written, and one byte less is refused."""
    from piper_kernels._hip import library as native

    h, tiles, last, sk, d, parts = case
    sq = (tiles - 1) * 128 + last
    log(f"[case] split workspace {case}")
    plan = MI355XPlan(waves=4, three_per_cu=True, key_parts=parts)
    lib = native.load_library()
    size = lib.attention_workspace_bytes(native.PiperShape(1, h, sq, sk, d), plan.plan_id)
    slots = torch.cuda.get_device_properties(gfx950_device).multi_processor_count * (4 if d == 64 else 3)
    first = h * tiles // slots * slots
    rows = h * sq - (first // tiles * sq + first % tiles * 128)
    key_tiles = -(-sk // 64)
    assert size == -(-key_tiles // -(-key_tiles // parts)) * rows * (d + 2) * 4
    g = torch.Generator().manual_seed(sq)
    q = torch.randn((1, h, sq, d), generator=g).to(torch.float16)
    k, v = (torch.randn((1, h, sk, d), generator=g).to(torch.float16) for _ in range(2))
    prepared = gpu_prepare(q, k, v, d**-0.5, False, gfx950_device, quantize_query=False, plan=plan)
    guarded = torch.full((size + 4096,), 0x5A, dtype=torch.uint8, device=gfx950_device)
    out = torch.empty((1, h, sq, d), device=gfx950_device)
    args = native.PiperAttentionFusedArgs(
        abi_version=native.ABI_VERSION, dtype=native.FLOAT16, output_dtype=native.FLOAT32, is_causal=0, plan=plan.plan_id,
        scale=d**-0.5, flags=0, reserved=0, shape=native.PiperShape(1, h, sq, sk, d),
        query=native.PiperTensor(prepared.query.data_ptr(), *prepared.query.stride()[:3]), prepared=prepared.native_prepared(),
        output=out.data_ptr(), workspace=guarded.data_ptr(), workspace_bytes=size - 1)
    stream = torch.cuda.current_stream(gfx950_device).cuda_stream
    with pytest.raises(RuntimeError, match="needs a workspace"):
        lib.attention_forward_fused(args, stream)
    args.workspace_bytes = size
    lib.attention_forward_fused(args, stream)
    torch.cuda.synchronize(gfx950_device)
    assert bool((guarded[size:] == 0x5A).all())
    assert torch.equal(out, gpu_attention(prepared, torch.float32))
