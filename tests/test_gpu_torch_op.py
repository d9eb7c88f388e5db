"""The native torch kernels (csrc/torch_op.cpp) against the Python path over the same C ABI: every option,
inputs read in place and inputs that must be copied, a side stream whose inputs are freed at once,
replays of a captured graph; errors stay Python exceptions; the plan source covers both operators."""

from __future__ import annotations

import importlib
import subprocess
import sys

import pytest
import torch

from _parity import log
from piper_kernels import piper_attention, sage_attention_2pp
from piper_kernels._hip import library as native
from piper_kernels._hip.build import PACKAGE_ROOT
from piper_kernels.attention.piper_attention import _plan
from piper_kernels.attention.piper_attention.hip import _run_piper_attention
from piper_kernels.attention.sage_attention_2pp.hip import _run_sage_attention_2pp

OPERATORS = {"piper": (piper_attention, _run_piper_attention), "sage": (sage_attention_2pp, _run_sage_attention_2pp)}


def _inputs(b, h, sq, sk, d, dtype, device, seed=0):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn((b, h, s, d), generator=g).to(dtype).to(device) for s in (sq, sk, sk))


@pytest.mark.gpu
@pytest.mark.parametrize("operator", OPERATORS)
@pytest.mark.parametrize("case", [
    # (B, H, Sq, Sk, D, dtype, causal, layout): layouts read in place (bhsd, bshd) or copied (odd)
    (1, 1, 1, 1, 64, torch.float16, False, "bhsd"),
    (2, 3, 77, 77, 128, torch.bfloat16, True, "bshd"),
    (1, 2, 300, 1000, 64, torch.bfloat16, False, "odd"),
    (1, 8, 1024, 1024, 64, torch.float16, False, "bhsd"),  # key-range split: a workspace
    (1, 24, 200, 3000, 128, torch.float16, False, "bshd"),
    (1, 5, 1100, 1100, 128, torch.bfloat16, True, "bshd"),  # causal key streams
], ids=str)
def test_native_call_equals_the_python_path(case, operator, gfx950_device) -> None:
    b, h, sq, sk, d, dtype, causal, layout = case
    log(f"[case] torch op {operator} {case}")
    q, k, v = _inputs(b, h, sq, sk, d, dtype, gfx950_device)
    if layout == "bshd":
        q, k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    elif layout == "odd":  # rows at odd multiples of two bytes
        q, k, v = (torch.cat([x, x[..., :1]], -1)[..., :d] for x in (q, k, v))
    public, python = OPERATORS[operator]
    with torch.no_grad():
        for scale in (None, 0.2):
            got = public(q, k, v, scale=scale, is_causal=causal)
            want = python(q, k, v, d**-0.5 if scale is None else scale, causal)
            assert got.is_contiguous() and got.dtype is dtype
            assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("operator", OPERATORS)
def test_streams_and_graph_replays(operator, gfx950_device) -> None:
    public, _ = OPERATORS[operator]
    log(f"[case] torch op streams and graph {operator}")
    sets = [_inputs(2, 4, 500, 500, 128, torch.float16, gfx950_device, seed) for seed in range(3)]
    with torch.no_grad():
        want = [public(*s, is_causal=True) for s in sets]
        side = torch.cuda.Stream(gfx950_device)
        side.wait_stream(torch.cuda.current_stream(gfx950_device))
        got = []
        for s in sets:
            copies = tuple(x.clone() for x in s)
            side.wait_stream(torch.cuda.current_stream(gfx950_device))
            with torch.cuda.stream(side):
                got.append(public(*copies, is_causal=True))
            del copies  # freed while the side stream may still read them
            torch.empty(1 << 20, device=gfx950_device).fill_(7.0)
        torch.cuda.synchronize(gfx950_device)
        assert all(torch.equal(a, b) for a, b in zip(got, want))

        static = tuple(x.clone() for x in sets[0])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = public(*static, is_causal=True)
        for i in (0, 1, 2, 0):
            for x, y in zip(static, sets[i]):
                x.copy_(y)
            graph.replay()
            torch.cuda.synchronize(gfx950_device)
            assert torch.equal(out, want[i]), f"replay {i}"
            assert torch.equal(public(*sets[i], is_causal=True), want[i])  # eager work between the replays


@pytest.mark.gpu
def test_errors_are_python_exceptions(gfx950_device) -> None:
    native.load_torch_kernels()
    op = torch.ops.piper_kernels.piper_attention
    q = torch.zeros((1, 1, 8, 32), dtype=torch.float16, device=gfx950_device)
    with pytest.raises(RuntimeError, match="head_dim must be 64 or 128"):
        op(q, q, q, 0.125, False)
    q = torch.zeros((1, 1, 8, 64), dtype=torch.float32, device=gfx950_device)
    with pytest.raises(RuntimeError, match="float16 or bfloat16"):
        op(q, q, q, 0.125, False)
    q = q.half()
    with pytest.raises(RuntimeError, match="scale must be finite and positive"):
        op(q, q, q, 0.0, False)


@pytest.mark.gpu
@pytest.mark.parametrize("operator", ["piper_attention", "sage_attention_2pp"])
def test_the_op_refuses_tensors_that_do_not_belong_together(operator, gfx950_device) -> None:
    """The kernels read key and value by the query's shape and type; nothing is launched here."""
    native.load_torch_kernels()
    op = getattr(torch.ops.piper_kernels, operator)
    q = torch.zeros((1, 2, 8, 64), dtype=torch.float16, device=gfx950_device)
    for key, value, text in [
        (q, q[:, :, :7], "key and value lengths match"),
        (q[:, :1], q[:, :1], "heads and head_dim must agree"),
        (q, q.bfloat16(), "share a dtype"),
        *([(q.bfloat16(), q.bfloat16(), "share a dtype")] if operator == "piper_attention" else []),
        (q.cpu(), q.cpu(), "share a device"),
        (q[0], q[0], "must have shape"),
    ]:
        with pytest.raises(RuntimeError, match=text):
            op(q, key, value, 0.125, False)


@pytest.mark.gpu
def test_sage_query_of_another_type_than_the_keys(gfx950_device) -> None:
    """Accepted by the op (the public function asks for one type): the output has the query's type."""
    native.load_torch_kernels()
    log("[case] torch op sage, fp16 query on bf16 keys")
    q, k, v = _inputs(1, 2, 100, 300, 64, torch.bfloat16, gfx950_device)
    with torch.no_grad():
        got = torch.ops.piper_kernels.sage_attention_2pp(q.half(), k, v, 0.125, False)
        assert got.dtype is torch.float16
        assert torch.equal(got, _run_sage_attention_2pp(q.half(), k, v, 0.125, False))


def test_plan_source_asks_the_package(monkeypatch) -> None:
    ask = native._choose_plan
    assert ask(0, 1, 8, 1024, 1024, 64, 0) == _plan.select_plan(1, 8, 1024, 1024, 64, False).plan_id
    assert ask(1, 4, 32, 8192, 8192, 128, 1) == _plan.select_sage_plan(4, 32, 8192, 8192, 128, True).plan_id
    monkeypatch.setattr(_plan, "select_plan", lambda *a: 1 / 0)
    assert ask(0, 1, 8, 1024, 1024, 64, 0) < 0  # an error in Python is no plan

    def interrupted(*_):
        raise KeyboardInterrupt

    monkeypatch.setattr(_plan, "select_plan", interrupted)
    assert ask(0, 1, 8, 1024, 1024, 64, 0) < 0  # and neither is an interrupt


@pytest.mark.gpu
def test_a_failed_plan_names_its_cause(gfx950_device, monkeypatch) -> None:
    def broken(*_):
        raise ValueError("this table has no such entry")

    q, k, v = _inputs(1, 1, 37, 41, 64, torch.float16, gfx950_device)  # a shape no other test plans
    monkeypatch.setattr(_plan, "select_plan", broken)
    with torch.no_grad(), pytest.raises(RuntimeError, match="ValueError: this table has no such entry"):
        piper_attention(q, k, v)
    monkeypatch.undo()
    with torch.no_grad():
        assert torch.isfinite(piper_attention(q, k, v)).all()


def test_kernels_are_registered_together_with_their_plan_source() -> None:
    """Opening the library registers nothing: a call of another thread between that and the plan source's
    setting would find kernels that cannot choose a plan."""
    program = """
import ctypes, sys
sys.path.insert(0, sys.argv[1])
import torch, piper_kernels
from piper_kernels._hip import library
from piper_kernels._hip.build import TORCH_LIBRARY_PATH
ops = ["piper_kernels::piper_attention", "piper_kernels::sage_attention_2pp"]
has = lambda: [torch._C._dispatch_has_kernel_for_dispatch_key(op, "CUDA") for op in ops]
kernels = ctypes.CDLL(str(TORCH_LIBRARY_PATH))
assert has() == [False, False], has()
library.load_torch_kernels()
assert has() == [True, True], has()
library.load_torch_kernels()
"""
    subprocess.run([sys.executable, "-c", program, str(PACKAGE_ROOT)], check=True, timeout=120)


@pytest.mark.gpu
def test_first_call_of_a_process_equals_the_next(gfx950_device) -> None:
    """A compiled graph, or the op itself, can be a process's first use; its bits are those of every later call
    (shapes that run key streams)."""
    log("[case] first call of a process")
    program = """
import sys
sys.path.insert(0, sys.argv[1])
import torch
from piper_kernels import piper_attention
g = torch.Generator().manual_seed(3)
q, k, v = (torch.randn((1, 3, 1000, 128), generator=g).to(torch.float16).cuda() for _ in range(3))
compiled = torch.compile(lambda q, k, v: piper_attention(q, k, v, is_causal=True), fullgraph=True, backend="eager")
with torch.no_grad():
    first = compiled(q, k, v)
    assert torch.equal(first, compiled(q, k, v)) and torch.equal(first, piper_attention(q, k, v, is_causal=True))
"""
    direct = """
import sys
sys.path.insert(0, sys.argv[1])
import torch, piper_kernels
op = torch.ops.piper_kernels.sage_attention_2pp
g = torch.Generator().manual_seed(4)
q, k, v = (torch.randn((1, 3, 1000, 128), generator=g).to(torch.float16).cuda() for _ in range(3))
assert torch.equal(op(q, k, v, 0.1, False), op(q, k, v, 0.1, False))
"""
    for text in (program, direct):
        subprocess.run([sys.executable, "-c", text, str(PACKAGE_ROOT)], check=True, timeout=100)


def _between_boundaries(x):
    """The same values in a contiguous view that starts two bytes after a 16-byte boundary."""
    return torch.cat([x.reshape(-1)[:1], x.reshape(-1)])[1:].view(x.shape)


def _odd_strides(x):
    """[1, 1, 1, D] values whose size-1 axes carry odd strides."""
    return torch.as_strided(x, x.shape, (7, 5, 3, 1))


@pytest.mark.parametrize("path", ["piper_attention", "sage_attention_2pp"])
def test_python_inputs_are_aligned_or_copied(path) -> None:
    module = importlib.import_module(f"piper_kernels.attention.{path}.hip")
    x = torch.randn(2, 3, 8, 64).half()
    got, arg = module._native_input(_between_boundaries(x))
    assert torch.equal(got, x) and arg.data == got.data_ptr() and arg.data % 16 == 0
    one = torch.randn(1, 1, 1, 64).half()
    got, arg = module._native_input(_odd_strides(one))
    assert got.data_ptr() == one.data_ptr() and (arg.stride_batch, arg.stride_head, arg.stride_seq) == (0, 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("operator", OPERATORS)
def test_contiguous_views_off_the_alignment_run(operator, gfx950_device) -> None:
    log(f"[case] torch op {operator} contiguous views between 16-byte boundaries, odd strides of size-1 axes")
    public, python = OPERATORS[operator]
    for view, shape in ((_between_boundaries, (2, 3, 77, 77)), (_odd_strides, (1, 1, 1, 1))):
        inputs = _inputs(*shape, 64, torch.float16, gfx950_device)
        with torch.no_grad():
            want = public(*inputs)
            assert torch.equal(public(*map(view, inputs)), want)
            assert torch.equal(python(*map(view, inputs), 64**-0.5, False), python(*inputs, 64**-0.5, False))
