"""catccos_amd._native_call: what reaches an entry point, and what is refused before it does."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from catccos_amd import _lib, _native_call, ops


@pytest.mark.parametrize("n", [0, 6, 7, 24])
def test_every_argument_arrives_in_its_place(n):
    got = []
    proto = C.CFUNCTYPE(C.c_int, *[C.c_uint64] * 24)

    @proto
    def callee(*args):
        got.extend(args)
        return -7
    values = [2 ** 40 + i if i % 3 else (None if i % 2 else -1 - i) for i in range(n)]
    assert _native_call.run(C.cast(callee, C.c_void_p).value, *values) == -7
    want = [0 if v is None else v % 2 ** 64 for v in values]
    assert got == want + [0] * (24 - n)


@pytest.mark.parametrize("value", [np.int64(2 ** 40 + 1), np.int32(-3), np.uint8(200), np.uint32(2 ** 32 - 1)], ids=lambda v: type(v).__name__)
def test_numpy_integers_are_integers(value):
    got = []
    proto = C.CFUNCTYPE(C.c_int, *[C.c_uint64] * 24)

    @proto
    def callee(*args):
        got.extend(args)
        return 0
    assert _native_call.run(C.cast(callee, C.c_void_p).value, 5, value, 6) == 0
    assert got[:4] == [5, int(value) % 2 ** 64, 6, 0]


def test_refusals():
    x = torch.zeros(2, 32, dtype=torch.bfloat16)
    address = _lib.entries()["cmx_version"]
    for args in ((address, x),):
        with pytest.raises(ValueError, match="expected a GPU tensor"):
            _native_call.run(*args)
    with pytest.raises(ValueError, match="expected a GPU tensor"):
        _native_call.empty(x, torch.uint8, 2)
    for call in (lambda: _native_call.run(), lambda: _native_call.run(address, *range(25)), lambda: _native_call.run(address, 1.5),
                 lambda: _native_call.run(address, "x"), lambda: _native_call.empty(x, torch.uint8), lambda: _native_call.empty(1, torch.uint8, 2)):
        with pytest.raises(TypeError):
            call()
    with pytest.raises(ValueError):
        _native_call.run(0, 1)
    for call in (lambda: ops.mx_quant(x), lambda: ops.mx_gemm(x, x, x, x, 32), lambda: ops.moe_init_routing(torch.zeros(2, 2, dtype=torch.int32), 4)):
        with pytest.raises(ValueError, match="expected a GPU tensor"):
            call()


def _host_calls():
    """Calls whose every buffer is the caller's, on host tensors: nothing that they allocate is refused before the call itself."""
    i32 = torch.zeros(2, dtype=torch.int32)
    a, s = torch.zeros(4, 128, dtype=torch.uint8), torch.zeros(4, 4, dtype=torch.uint8)
    b, bs = torch.zeros(2, 64, 128, dtype=torch.uint8), torch.zeros(2, 64, 4, dtype=torch.uint8)
    work = torch.zeros(4096, dtype=torch.uint8)
    return {"mx_gmm": lambda: ops.mx_gmm(a, s, b, bs, i32, 128, c=torch.zeros(4, 64, dtype=torch.bfloat16), workspace=work),
            "mx_gmm, its own buffers": lambda: ops.mx_gmm(a, s, b, bs, i32, 128),
            "mx_gmm_swiglu_quant": lambda: ops.mx_gmm_swiglu_quant(a, s, b, bs, i32, 128, workspace=work,
                                                                   outs=(torch.zeros(4, 32, dtype=torch.uint8), torch.zeros(4, 2, dtype=torch.uint8))),
            "int8_gmm_dequant_swiglu": lambda: ops.int8_gmm_dequant_swiglu(a.view(torch.int8), torch.zeros(4), b.view(torch.int8), torch.zeros(128), i32,
                                                                           64, 128, 1, c=torch.zeros(4, 32))}


@pytest.mark.parametrize("name", _host_calls())
def test_host_tensors_are_refused_as_such(name):
    # also in a process without a GPU, where asking for the current stream would fail first
    with pytest.raises(ValueError, match="expected a GPU tensor"):
        _host_calls()[name]()


def test_the_front_end_imports_without_the_extension():
    """The extension is asked for by the first call that needs it; its absence is an ImportError that says how to build it."""
    code = """
import sys
sys.modules["catccos_amd._native_call"] = None              # an import of it fails
import torch
from catccos_amd import ops
assert ops.scale_cols(96) == 4 and ops.ffn_workspace_bytes(1, 256, 512, 2, 1) > 0
for _ in range(2):
    try:
        ops.mx_quant(torch.zeros(2, 32, dtype=torch.bfloat16))
    except ImportError as e:
        assert "python -m catccos_amd.build" in str(e)
    else:
        raise AssertionError("no ImportError")
del sys.modules["catccos_amd._native_call"]                 # built in the meantime
try:
    ops.mx_quant(torch.zeros(2, 32, dtype=torch.bfloat16))
except ValueError:
    print("ok")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=root, timeout=110)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stderr


def test_the_extension_is_rebuilt_for_another_torch(monkeypatch, tmp_path):
    """Newer than its source is not enough: a change of torch or of the command builds it again; a failed build leaves the old one alone."""
    from catccos_amd import build
    target, calls = tmp_path / "ext.so", []

    def compiler(cmd, **kw):
        calls.append(cmd)
        out = cmd[cmd.index("-o") + 1]
        with open(out, "w") as f:
            f.write(f"build {len(calls)}")
        return subprocess.CompletedProcess(cmd, 1 if len(calls) == 3 else 0, "", "error")
    monkeypatch.setattr(build, "NATIVE", str(target))
    monkeypatch.setattr(build, "OBJ", str(tmp_path / "obj"))
    monkeypatch.setattr(build.subprocess, "run", compiler)
    build.build_native()
    build.build_native()
    assert len(calls) == 1 and target.read_text() == "build 1"
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    build.build_native()
    build.build_native()
    assert len(calls) == 2 and target.read_text() == "build 2"
    with pytest.raises(RuntimeError, match="error"):
        build.build_native(force=True)
    assert target.read_text() == "build 2" and sorted(os.listdir(tmp_path)) == ["ext.so", "obj"]


def test_an_extension_of_another_torch_is_refused(monkeypatch):
    assert _native_call.torch_version == torch.__version__
    monkeypatch.setattr(_native_call, "torch_version", "0.0.0")
    with pytest.raises(ImportError, match="built for torch 0.0.0"):
        ops._bind_native()


@pytest.mark.parametrize("name, call", [
    ("cmx_mx_gemm", lambda x, i32, n: ops.mx_gemm(x, x, x, x, n(32))),
    ("cmx_mx_gemm_ex", lambda x, i32, n: ops.mx_gemm_ex(x, x, x, x, n(2), n(3), n(64), trans_a=n(0), trans_b=n(1))),
    ("cmx_int8_quant_scatter", lambda x, i32, n: ops.int8_quant_scatter(x, i32, n(4))),
    ("cmx_int8_gmm_dequant_swiglu", lambda x, i32, n: ops.int8_gmm_dequant_swiglu(x, x, x, x, i32, n(64), n(128), n(1), scale_stride=n(5), c=x)),
    ("cmx_mx_gmm", lambda x, i32, n: ops.mx_gmm(x, x, x, x, i32, n(32), c=x, workspace=x)),
    ("cmx_mx_gmm_swiglu_quant", lambda x, i32, n: ops.mx_gmm_swiglu_quant(x, x, x, x, i32, n(32), outs=(x, x), workspace=x)),
    ("cmx_moe_init_routing", lambda x, i32, n: ops.moe_init_routing(i32.view(1, 2), n(7))),
    ("cmx_quant_scatter_zeroed", lambda x, i32, n: ops.quant_scatter(x, i32, n(4)))])
def test_whole_numbers_as_tensors_of_one_element(monkeypatch, name, call):
    """A size or flag given as a tensor of one element (which converts to an index) reaches the entry point as the number."""
    seen = []

    def run(address, *args):
        seen.append([a for a in args if not isinstance(a, torch.Tensor)])
        return 0
    monkeypatch.setattr(ops, "_run", run)
    monkeypatch.setattr(ops, "_empty", lambda like, dtype, *size: torch.empty(*(int(v) for v in size), dtype=dtype))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_need_cuda", lambda *ts: None)
    monkeypatch.setattr(_lib, "entries", lambda: {name: 1})
    x, i32 = torch.zeros(2, 32, dtype=torch.bfloat16), torch.zeros(2, dtype=torch.int32)
    call(x, i32, int)
    call(x, i32, torch.tensor)
    assert seen[0] == seen[1] and len(seen) == 2, seen


def test_entries_follow_the_active_library():
    before = _lib.entries()
    prev = _lib.activate(None)
    try:
        assert _lib.entries() is not before
    finally:
        _lib.activate(prev)
    assert set(_lib.entries()) == set(_lib.SIGNATURES) and all(_lib.entries().values())


def test_an_ellipsis_in_the_place_of_a_tensor_is_refused():
    """Only the front end puts one, behind the other arguments; one that the caller gives would leave a null pointer in its place."""
    got = []

    @C.CFUNCTYPE(C.c_int, *[C.c_uint64] * 24)
    def callee(*args):
        got.append(args)
        return 0
    with pytest.raises(TypeError, match="Ellipsis"):
        _native_call.run(C.cast(callee, C.c_void_p).value, ..., 1, ...)
    assert not got


def test_a_tuple_in_the_place_of_a_tensor_is_refused():
    """Only the front end puts one, for a new tensor; one that the caller gives would reach the kernel as a tensor of anything."""
    spec, x = (torch.int32, 8), torch.zeros((8, 64), dtype=torch.bfloat16)
    with pytest.raises(TypeError, match="tuple"):
        ops.int8_quant_scatter(x, spec, 1)
    a, w, scale, sizes = x.view(torch.int16).to(torch.int8), torch.zeros((1, 64, 64), dtype=torch.int8), torch.ones(64), torch.zeros(1, dtype=torch.int32)
    for token, channel in (spec, scale), (scale, spec):
        with pytest.raises(TypeError, match="tuple"):
            ops.int8_gmm_dequant_swiglu(a, token, w, channel, sizes, 64, 64, 1)


@pytest.mark.gpu
def test_outputs_and_errors_on_the_gpu():
    x = torch.randn(3, 64, device="cuda").to(torch.bfloat16)
    t = _native_call.empty(x, torch.float16, 2, 3, 4)
    assert t.shape == (2, 3, 4) and t.dtype == torch.float16 and t.device == x.device and not t.requires_grad
    assert _native_call.empty(x, torch.uint8, 0).numel() == 0
    with pytest.raises(_lib.CmxError, match="k must be"):
        ops.mx_gemm(x.view(torch.uint8), x.view(torch.uint8), x.view(torch.uint8), x.view(torch.uint8), 33)
    with pytest.raises(ValueError, match="expected a GPU tensor"):
        ops.mx_gemm(x.view(torch.uint8), x.view(torch.uint8), x.view(torch.uint8).cpu(), x.view(torch.uint8), 32)


@pytest.mark.gpu
def test_new_tensors_and_the_current_stream_reach_the_entry_point():
    got, rc = [], [0]
    proto = C.CFUNCTYPE(C.c_int, *[C.c_uint64] * 24)

    @proto
    def callee(*args):
        got.append(args)
        return rc[0]
    address = C.cast(callee, C.c_void_p).value
    x = torch.zeros(4, device="cuda")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        a, b = _native_call.run(address, 1, (torch.uint8, 3, 5), x, (torch.float32, 7), ...)
    assert a.shape == (3, 5) and a.dtype == torch.uint8 and b.shape == (7,) and b.dtype == torch.float32 and a.device == b.device == x.device
    assert got[0][:6] == (1, a.data_ptr(), x.data_ptr(), b.data_ptr(), side.cuda_stream, 0)
    one = _native_call.run(address, x, (torch.int32, 2, 0), ...)
    assert one.shape == (2, 0) and got[1][2] == torch.cuda.current_stream().cuda_stream
    rc[0] = -5
    assert _native_call.run(address, x, (torch.uint8, 1)) == -5
    for bad in (lambda: _native_call.run(address, x, ("u8", 1)), lambda: _native_call.run(address, x, (torch.uint8,)),
                lambda: _native_call.run(address, x, *[(torch.uint8, 1)] * 5)):
        with pytest.raises(TypeError):
            bad()
    with pytest.raises(ValueError, match="expected a GPU tensor"):
        _native_call.run(address, 1, (torch.uint8, 1))
    with pytest.raises(RuntimeError):
        _native_call.run(address, x, (torch.uint8, -2))
    assert len(got) == 3


@pytest.mark.gpu
def test_new_tensors_are_those_of_torch_empty():
    """Filled where deterministic algorithms are asked for, seen by a dispatch mode, inference tensors in inference mode."""
    from torch.utils._python_dispatch import TorchDispatchMode
    x = torch.zeros(4, device="cuda")
    routes = torch.tensor([[0, -1], [7, 1]], dtype=torch.int32, device="cuda")          # two of four dropped
    was = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True)
    try:
        assert bool(_native_call.empty(x, torch.float32, 5, 3).isnan().all())
        assert ops.moe_init_routing(routes, 2)[0].tolist() == [0, 3, 2 ** 31 - 1, 2 ** 31 - 1]
    finally:
        torch.use_deterministic_algorithms(was)

    class Seen(TorchDispatchMode):
        def __init__(self, give=None):
            super().__init__()
            self.calls, self.give = [], give

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.calls.append(func)
            return func(*args, **(kwargs or {})) if self.give is None else self.give
    with Seen() as mode:
        ops.moe_init_routing(routes, 2)
    assert mode.calls == [torch.ops.aten.empty.memory_format] * 4                       # workspace and three outputs
    with Seen(torch.zeros(5)), pytest.raises(ValueError, match="expected a GPU tensor"):
        _native_call.empty(x, torch.float32, 5)
    with torch.inference_mode():
        assert ops.moe_init_routing(routes, 2)[2].is_inference()
    assert not ops.moe_init_routing(routes, 2)[2].is_inference()


@pytest.mark.gpu
def test_buffers_that_the_caller_brings_may_be_pinned():
    """Weights, outputs and workspaces in pinned host memory give the results that device buffers give (no kernel of these small problems uses
    the workspace); other host memory, and inputs in host memory, are refused."""
    gen = torch.Generator().manual_seed(3)
    u8 = lambda *shape, hi=0x70: torch.randint(0, hi, shape, dtype=torch.uint8, generator=gen)
    m, k, n, sizes = 96, 256, 128, torch.tensor([40, 0, 50], dtype=torch.int32).cuda()
    a, s = u8(m, k).cuda(), (u8(m, 8, hi=8) + 120).cuda()
    b, bs = u8(3, n, k), (u8(3, n, 8, hi=8) + 120).cuda()
    work = ops.gmm_workspace(3, "cuda")
    pinned = lambda *shape, dtype=torch.uint8: torch.zeros(shape, dtype=dtype, pin_memory=True)

    want = ops.mx_gmm(a, s, b.cuda(), bs, sizes, k)
    c = pinned(m, n, dtype=torch.bfloat16)
    ops.mx_gmm(a, s, b.pin_memory(), bs, sizes, k, c=c, workspace=work)
    codes, scales, _ = ops.mx_gmm_swiglu_quant(a, s, b.cuda(), bs, sizes, k)
    outs = pinned(m, n // 2), pinned(m, 2)
    ops.mx_gmm_swiglu_quant(a, s, b.pin_memory(), bs, sizes, k, workspace=pinned(work.numel()), outs=outs)
    i8 = lambda t: t.view(torch.int8)
    token, channel = torch.rand(m, generator=gen).cuda(), torch.rand(3 * n, generator=gen).cuda()
    want8 = ops.int8_gmm_dequant_swiglu(i8(a), token, i8(b).cuda(), channel, sizes, n, k, 1)
    c8 = pinned(m, n // 2, dtype=torch.float32)
    ops.int8_gmm_dequant_swiglu(i8(a), token, i8(b).cuda(), channel, sizes, n, k, 1, c=c8)
    torch.cuda.synchronize()
    assert torch.equal(c, want.cpu()) and want.float().abs().max() > 0
    assert torch.equal(outs[0], codes.cpu()) and torch.equal(outs[1], scales.cpu())
    assert torch.equal(c8, want8.cpu())

    for call in (lambda: ops.mx_gmm(a, s, b.cuda(), bs, sizes, k, c=torch.zeros(m, n, dtype=torch.bfloat16), workspace=work),
                 lambda: ops.mx_gmm(a, s, b, bs, sizes, k), lambda: ops.mx_gmm(a, s.cpu().pin_memory(), b.cuda(), bs, sizes, k),
                 lambda: ops.int8_gmm_dequant_swiglu(i8(a), token, i8(b).pin_memory(), channel, sizes, n, k, 1)):
        with pytest.raises(ValueError, match="expected a GPU tensor"):
            call()
