"""The persistent 256 x 256 kernels with 2 x 2 wavefronts: their walk through more and less than whole rounds of tiles, groups found by a
scan of the sizes, and the INT8 kernel.  Reference: the streaming kernel of the same tile, one tile per workgroup, whose K order (INT8:
whole-number sums) is the same, so the outputs are the same bits."""
import ctypes

import numpy as np
import pytest
import torch

from tests.gpu_util import dev, hooked_library, hooks_lib

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _hooked():
    with hooked_library():
        yield


def _pinned(call):
    """call() with the persistent kernels and with the streaming ones"""
    h = hooks_lib()
    h.cmx_debug_force_ksplit(-1, 0, 0)
    h.cmx_debug_force_tile(256, 256, 4)
    got = call()
    h.cmx_debug_force_tile(256, 256, 8)
    return got, call()


# tiles: less than a round; 1 + 64 tiles, 2 + 200 and 3 + 8 rounds of 256
ROUNDS = [([300, 0, 257, 1], 512), ([640] * 8 + [0, 3], 2560), ([520] * 16 + [0, 513, 9], 3072), ([256] * 97, 2048)]


@pytest.mark.parametrize("counts,n", ROUNDS)
@pytest.mark.parametrize("kind", ["SwiGLU", "E2M1", "dense"])
def test_walk_through_rounds(kind, counts, n):
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    e, m, k = len(counts), sum(counts) + 5, 512
    kb = k // 2 if kind == "E2M1" else k
    codes = lambda *shape: torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xF7
    scales = lambda *shape: torch.randint(110, 125, shape, dtype=torch.uint8, device="cuda", generator=g)
    a, a_s, w, w_s = codes(m, kb), scales(m, k // 32), codes(e, n, kb), scales(e, n, k // 32)
    cnt = dev(np.array(counts, dtype=np.int32))

    def call():
        if kind == "SwiGLU":
            outs = torch.full((m, n // 2), 7, dtype=torch.uint8, device="cuda"), torch.full((m, ops.scale_cols(n // 2)), 7, dtype=torch.uint8, device="cuda")
            return ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k, outs=outs)[:2]
        if kind == "E2M1":
            return [ops.mx_gmm(a, a_s, w, w_s, cnt, k, "E2M1", c=torch.full((m, n), 7.0, dtype=torch.bfloat16, device="cuda"))]
        return [ops.mx_gemm(a, a_s, w[0], w_s[0], k)]
    for got, ref in zip(*_pinned(call)):
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8)) and bool((ref != 7).any())


@pytest.mark.parametrize("sizes,rows", [([5, -3, 0, 700, 1], 706), ([40, 2 ** 31 - 1, 2 ** 31 - 1, 9], 300), ([0, 0, 0], 10), ([1] * 256, 256),
                                        ([300, 0, 66, 1] * 64, 23000)])
@pytest.mark.parametrize("kind", ["SwiGLU", "E2M1", "INT8"])
def test_scanned_groups_are_those_of_the_tables(kind, sizes, rows):
    """Up to 256 groups are scanned, more go through tables: empty groups behind the last one change nothing."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    n, k, many = 64, 512, 300
    kb = k // 2 if kind == "E2M1" else k
    codes = lambda *shape: torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xF7
    a, w = codes(rows, kb), codes(many, n, kb)
    a_s, w_s = (torch.randint(110, 125, s, dtype=torch.uint8, device="cuda", generator=g) for s in ((rows, k // 32), (many, n, k // 32)))
    h = hooks_lib()
    h.cmx_debug_force_ksplit(-1, 0, 0)
    h.cmx_debug_force_tile(256, 256, 4)

    def outputs(counts):
        e, cnt = len(counts), dev(np.array(counts, dtype=np.int32))
        if kind == "INT8":
            return [ops.int8_gmm_dequant_swiglu(a.view(torch.int8), torch.ones(rows, device="cuda"), w[:e].view(torch.int8),
                                                torch.full((e * n,), 1e-5, device="cuda"), cnt, n, k, 1, c=torch.zeros((rows, n // 2), device="cuda"))]
        if kind == "SwiGLU":
            outs = torch.zeros((rows, n // 2), dtype=torch.uint8, device="cuda"), torch.zeros((rows, 2), dtype=torch.uint8, device="cuda")
            return ops.mx_gmm_swiglu_quant(a, a_s, w[:e], w_s[:e], cnt, k, outs=outs)[:2]
        return [ops.mx_gmm(a, a_s, w[:e], w_s[:e], cnt, k, "E2M1", c=torch.zeros((rows, n), dtype=torch.bfloat16, device="cuda"))]
    for got, want in zip(outputs(sizes), outputs(sizes + [0] * (many - len(sizes)))):
        assert torch.equal(got, want) and (bool((got != 0).any()) or sum(sizes) == 0)


# K of two slabs, of odd numbers of slabs and of whole blocks; a quarter of a tile along n, a tile and a half, whole ones; 300 groups (tables)
@pytest.mark.parametrize("counts,n,k", [([300, 0, 257, 1], 64, 256), ([256] * 3 + [5], 384, 384), ([512, 31], 256, 1024),
                                        ([700] * 40, 768, 640), ([1300, 0, 900] * 8, 2560, 128 * 9), ([290, 3] * 150, 128, 512)])
@pytest.mark.parametrize("out", ["fp32", "bf16", "fp16"])
def test_int8_gives_the_bits_of_the_streaming_kernel(out, counts, n, k):
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    e, m = len(counts), sum(counts)
    dtype = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[out]
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (e, n, k), dtype=torch.int8, device="cuda", generator=g)
    channel, token = torch.rand(e * n * 2, device="cuda", generator=g) * 1e-4, torch.rand(m, device="cuda", generator=g)
    cnt = dev(np.array(counts, dtype=np.int32))

    def call():
        c = torch.full((m + 3, n // 2), 7.0, dtype=dtype, device="cuda")
        ops.int8_gmm_dequant_swiglu(a, token, w, channel, cnt, n, k, 1, out, scale_stride=2, c=c[:m])
        assert bool((c[m:] == 7.0).all())
        return c
    got, ref = _pinned(call)
    assert torch.equal(got, ref) and not bool((ref[:m] == 7.0).all(dim=1).any())


@pytest.mark.parametrize("out", ["fp32", "bf16", "fp16"])
def test_int8_rounds_special_values_like_the_streaming_kernel(out):
    """Token scales that make outputs zero, denormal, halfway between neighbours, infinite and NaN."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    counts, n, k = [256, 300], 256, 512
    m = sum(counts)
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (2, n, k), dtype=torch.int8, device="cuda", generator=g)
    w[:, 0], w[:, n // 2] = 0, 0                                                     # sums of zero, which infinite scales make NaN
    token = torch.rand(m, device="cuda", generator=g)
    special = [0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1e-38, 1e-42, 1e-20, 2.0 ** -12, 2.0 ** -13, 3.0, 1e4, 1e30, 3e38]
    token[:16 * len(special)] = torch.tensor(special, device="cuda").repeat(16)
    token[-1], token[-2] = torch.tensor([0x7F80_0001, -1], dtype=torch.int32).view(torch.float32).cuda()            # other NaNs
    channel = torch.full((2 * n,), 2.0 ** -10, device="cuda")
    channel[::7] = torch.rand(channel[::7].numel(), device="cuda", generator=g)
    call = lambda: ops.int8_gmm_dequant_swiglu(a, token, w, channel, dev(np.array(counts, dtype=np.int32)), n, k, 1, out)
    got, ref = _pinned(call)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16)) and bool(ref.isnan().any()) and bool(ref.isinf().any())


class _KernelNode(ctypes.Structure):
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _kernels_of(call):
    """the kernels that a call launches, in no order, read from a capture of it"""
    hip = ctypes.CDLL("libamdhip64.so")
    call()                                             # (limits of the LDS are raised at the first launch)
    graph, n = torch.cuda.CUDAGraph(keep_graph=True), ctypes.c_size_t()
    with torch.cuda.graph(graph):
        call()
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        k = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(k)) == 0
        out.append(k.func)
    return sorted(out)


# at most two rounds of tiles: an odd number of slabs, one past the K up to which it counts, even; short groups; 16-bit output; past two rounds
@pytest.mark.parametrize("e,rows,n,k,out,waves", [(16, 300, 2048, 384, "fp32", 8), (16, 300, 2048, 1920, "fp32", 8), (16, 300, 2048, 2176, "fp32", 4), (16, 300, 2048, 512, "fp32", 4),
                                                  (16, 300, 2048, 256, "fp32", 8), (32, 140, 2048, 1536, "fp32", 8), (32, 140, 2048, 1792, "fp32", 4), (16, 300, 2048, 384, "bf16", 4),
                                                  (8, 1900, 2048, 384, "fp32", 4)])
def test_int8_kernel_by_size(e, rows, n, k, out, waves):
    """waves: 8 the streaming kernel, 4 the persistent one"""
    from catccos_amd import ops
    a, w = torch.zeros((e * rows, k), dtype=torch.int8, device="cuda"), torch.zeros((e, n, k), dtype=torch.int8, device="cuda")
    token, channel, cnt = torch.ones(e * rows, device="cuda"), torch.ones(e * n, device="cuda"), dev(np.full(e, rows, dtype=np.int32))
    c = torch.empty((e * rows, n // 2), dtype=torch.float32 if out == "fp32" else torch.bfloat16, device="cuda")
    call = lambda: ops.int8_gmm_dequant_swiglu(a, token, w, channel, cnt, n, k, 1, out, c=c)
    h = hooks_lib()
    h.cmx_debug_force_ksplit(-1, 0, 0)
    got, pinned = _kernels_of(call), {}
    for v in (4, 8):
        h.cmx_debug_force_tile(256, 256, v)
        pinned[v] = _kernels_of(call)
    assert pinned[4][-1:] != pinned[8][-1:] and got == pinned[waves]


# 8-bit SwiGLU in groups of at most 128 rows: the ring kernel, but for many rounds of its tiles at K below 1536
@pytest.mark.parametrize("e,rows,n,k,waves", [(256, 40, 2048, 1024, 5), (256, 40, 2048, 1408, 5), (256, 40, 2048, 1536, 6), (160, 40, 2048, 1024, 6), (32, 100, 2048, 1024, 6)])
def test_swiglu_kernel_of_short_groups_by_size(e, rows, n, k, waves):
    """waves: 5 the three-slot kernel, 6 the ring kernel"""
    from catccos_amd import ops
    z = lambda *shape: torch.zeros(shape, dtype=torch.uint8, device="cuda")
    a, a_s, w, w_s, cnt = z(e * rows, k), z(e * rows, k // 32), z(e, n, k), z(e, n, k // 32), dev(np.full(e, rows, dtype=np.int32))
    outs, ws = (z(e * rows, n // 2), z(e * rows, ops.scale_cols(n // 2))), ops.gmm_workspace(e, "cuda")
    call = lambda: ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k, workspace=ws, outs=outs)
    h = hooks_lib()
    h.cmx_debug_force_ksplit(-1, 0, 0)
    got, pinned = _kernels_of(call), {}
    for v in (5, 6):
        h.cmx_debug_force_tile(256, 128, v)
        pinned[v] = _kernels_of(call)
    assert pinned[5] != pinned[6] and got == pinned[waves]
