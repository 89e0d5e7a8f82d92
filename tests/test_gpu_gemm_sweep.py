"""Seeded shape sweeps of the dense and grouped matmuls against the oracle.  Sizes this small go to the split-K kernels (dense) or, by
the average rows per group, to those and the 256-row kernels (grouped); the dense sweep runs a second time with split-K switched
off, which takes the same sizes through the kernels behind it (hand-scheduled two- and three-slot, streaming,
register-staged).  Dense problems large enough for these in the product library are in test_dense_past_split_k."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as O
from tests.gpu_util import dev, host, close_bf16, hooked_library

pytestmark = pytest.mark.gpu


def _shapes(seed, count):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        m = int(rng.choice([1, 17, 64, 100, 128, 129, 255, 256, 257, 300, 511, 600, 777]))
        n = int(rng.choice([4, 32, 100, 256, 260, 512, 700, 1028]))
        k = int(rng.choice([32, 96, 128, 256, 384, 512, 768, 1024, 2048]))
        out.append((m, n, k))
    return out


@pytest.mark.parametrize("split_k", [True, False])
@pytest.mark.parametrize("m,n,k", _shapes(1, 36))
def test_dense_sweep(m, n, k, split_k):
    from catccos_amd import ops
    rng = np.random.default_rng(m * 131 + n * 17 + k)
    aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m, k)).astype(np.float32)), "E4M3")
    bq, bsc = O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), "E4M3")
    if split_k:
        c = ops.mx_gemm(dev(aq), dev(asc), dev(bq), dev(bsc), k)
    else:
        with hooked_library() as lib:
            lib.cmx_debug_force_ksplit(-1, 0, 0)
            c = ops.mx_gemm(dev(aq), dev(asc), dev(bq), dev(bsc), k)
    bad, worst = close_bf16(host(c), O.mx_gemm_f32(aq, asc, bq, bsc))
    assert bad == 0, (bad, worst)


def _past_split_k(m, n, k):
    """More 64 x 64 tiles than the library gives to the split-K kernels (four per CU, eight where K is no whole number of
    slabs), and more 128 x 128 tiles than CUs."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return -(-m // 64) * -(-n // 64) > (4 if k % 128 == 0 else 8) * cus and -(-m // 128) * -(-n // 128) > cus


@pytest.mark.parametrize("fmt,out,m,n,k", [
    ("E4M3", "bf16", 2100, 4104, 1024), ("E4M3", "fp16", 2100, 4104, 1024), ("E5M2", "fp16", 2049, 4112, 512),      # persistent, whole-line stores
    ("E4M3", "fp32", 2100, 4104, 512), ("E4M3", "bf16", 2100, 4100, 512),                                            # two-slot, one tile per workgroup
    ("E4M3", "bf16", 2100, 4104, 640), ("E5M2", "bf16", 2050, 4104, 96),                                             # streaming; register-staged
    ("E2M1", "bf16", 2100, 4104, 1024), ("E2M1", "fp16", 2100, 4104, 512), ("E2M1", "fp32", 2100, 4104, 512), ("E2M1", "bf16", 2100, 4104, 768)])
def test_dense_past_split_k(fmt, out, m, n, k):
    """The 256-row kernels as the product library compiles and chooses them, with a ragged last row tile and a ragged last column
    tile (n % 256 = 4, 8 or 16)."""
    from catccos_amd import ops
    assert _past_split_k(m, n, k)
    rng = np.random.default_rng(m + n + k)
    aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m, k)).astype(np.float32)), fmt)
    bq, bsc = O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), fmt)
    pack = O.pack_fp4 if fmt == "E2M1" else (lambda x: x)
    gold = O.mx_dequant(aq, asc, fmt).astype(np.float32) @ O.mx_dequant(bq, bsc, fmt).astype(np.float32).T
    c = host(ops.mx_gemm(dev(pack(aq)), dev(asc), dev(pack(bq)), dev(bsc), k, fmt, out))
    if out == "bf16":
        bad, worst = close_bf16(c, gold)
        assert bad == 0, (bad, worst)
    else:
        # as for the smaller problems: 8-bit products keep 2^-13 of the largest of eight, FP4 products are exact
        rtol, atol = (1e-3, 1e-2) if fmt != "E2M1" else (1e-5, 1e-3)
        if out == "fp16":
            rtol, atol = rtol + 2.0 ** -11, atol + 2.0 ** -11
        assert np.allclose(c.astype(np.float64), gold, rtol=rtol, atol=atol), np.abs(c - gold).max()


def _groupings(seed, count):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        g = int(rng.integers(1, 9))
        scale = int(rng.choice([8, 70, 140, 300, 520]))
        counts = [int(c) for c in rng.integers(0, scale + 1, size=g)]
        if sum(counts) == 0:
            counts[0] = 3
        n = int(rng.choice([64, 256, 320, 768]))
        k = int(rng.choice([128, 256, 512, 1024]))
        out.append((tuple(counts), n, k))
    return out


@pytest.mark.parametrize("counts,n,k", _groupings(2, 24))
def test_grouped_sweep(counts, n, k):
    from catccos_amd import ops
    rng = np.random.default_rng(sum(counts) * 7 + n + k)
    m = sum(counts)
    aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m, k)).astype(np.float32)))
    ws_ = [O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), "E4M3", "lut") for _ in counts]
    wq, ws = np.stack([q for q, _ in ws_]), np.stack([s for _, s in ws_])
    cnt = dev(np.array(counts, dtype=np.int32))
    c = ops.mx_gmm(dev(aq), dev(asc), dev(wq), dev(ws), cnt, k)
    bad, worst = close_bf16(host(c), O.mx_gmm_f32(aq, asc, wq, ws, list(counts)))
    assert bad == 0, (bad, worst)
    if n % 64 == 0:
        # fused SwiGLU + requant on the same operands: dequantised activation within the bound of two chained
        # bf16 roundings and one E4M3 quantisation step
        codes, scales, _ = ops.mx_gmm_swiglu_quant(dev(aq), dev(asc), dev(wq), dev(ws), cnt, k)
        _, _, gq, gs = O.gmm1_swiglu_quant(aq, asc, wq, ws, list(counts))
        deq, deq_g = O.mx_dequant(host(codes), host(scales)), O.mx_dequant(gq, gs)
        bound = 0.13 * np.abs(deq_g) + 2.0 ** -5 * np.abs(deq_g).max(axis=1, keepdims=True) + 1e-6
        assert np.all(np.abs(deq - deq_g) <= bound)


@pytest.mark.parametrize("fmt", ["E4M3", "E2M1"])
@pytest.mark.parametrize("out", ["bf16", "fp16"])
@pytest.mark.parametrize("m,n", [(300, 520), (2100, 4104)])
def test_output_pitch_and_edges_are_left_alone(fmt, out, m, n):
    """300 x 520: the split-K kernel; 2100 x 4104: the persistent kernels, which store their 16-bit output in whole lines through the
    LDS.  With an output pitch wider than n, a ragged last row tile and a ragged last column tile, every element inside
    equals the tight-pitch call bit for bit and every element outside keeps its poison."""
    from catccos_amd import _lib, ops
    k, ldc, pad_rows = 1024, n + 16, 3
    assert _past_split_k(m, n, k) == (m > 300)
    rng = np.random.default_rng(77)
    if fmt == "E2M1":
        aq, asc = O.mx_quant(rng.uniform(-2, 2, (m, k)).astype(np.float32), "E2M1")
        bq, bsc = O.mx_quant(rng.uniform(-2, 2, (n, k)).astype(np.float32), "E2M1")
        aq, bq = O.pack_fp4(aq), O.pack_fp4(bq)
    else:
        aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m, k)).astype(np.float32)), "E4M3")
        bq, bsc = O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), "E4M3")
    a, a_s, b, b_s = dev(aq), dev(asc), dev(bq), dev(bsc)
    tight = ops.mx_gemm(a, a_s, b, b_s, k, fmt, out)
    wide = torch.full((m + pad_rows, ldc), 0x7FC1, dtype=torch.int16, device="cuda")
    lib = _lib.load()
    _lib.check(lib.cmx_mx_gemm(a.data_ptr(), a.stride(0), a_s.data_ptr(), a_s.stride(0), b.data_ptr(), b.stride(0), b_s.data_ptr(),
                               b_s.stride(0), wide.data_ptr(), ldc, m, n, k, ops.FMT[fmt], ops.OUT[out],
                               torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(wide[:m, :n], tight.view(torch.int16))
    assert bool((wide[:m, n:] == 0x7FC1).all()) and bool((wide[m:] == 0x7FC1).all())


@pytest.mark.parametrize("fmt", ["E4M3", "E2M1"])
def test_grouped_output_pitch_and_edges_are_left_alone(fmt):
    """The same for the grouped matmul (ragged groups, one empty, rows past the groups): inside bit-equal to the
    tight-pitch call, outside untouched."""
    from catccos_amd import ops
    counts, n, k, ldc, spare = [700, 0, 900, 650], 520, 1024, 536, 5
    m = sum(counts)
    rng = np.random.default_rng(78)
    if fmt == "E2M1":
        aq, asc = O.mx_quant(rng.uniform(-2, 2, (m + spare, k)).astype(np.float32), "E2M1")
        ws_ = [O.mx_quant(rng.uniform(-2, 2, (n, k)).astype(np.float32), "E2M1") for _ in counts]
        aq = O.pack_fp4(aq)
        wq = np.stack([O.pack_fp4(q) for q, _ in ws_])
    else:
        aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m + spare, k)).astype(np.float32)), "E4M3")
        ws_ = [O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), "E4M3", "lut") for _ in counts]
        wq = np.stack([q for q, _ in ws_])
    wsc = np.stack([s for _, s in ws_])
    a, a_s, w, w_s = dev(aq), dev(asc), dev(wq), dev(wsc)
    cnt = torch.tensor(counts, dtype=torch.int32, device="cuda")
    tight = ops.mx_gmm(a, a_s, w, w_s, cnt, k, fmt)
    wide = torch.full((m + spare, ldc), 0x7FC1, dtype=torch.int16, device="cuda")
    ops.mx_gmm(a, a_s, w, w_s, cnt, k, fmt, c=wide.view(torch.bfloat16)[:, :n])
    torch.cuda.synchronize()
    assert torch.equal(wide[:m, :n], tight.view(torch.int16)[:m])
    assert bool((wide[:, n:] == 0x7FC1).all()) and bool((wide[m:] == 0x7FC1).all())
