"""The ring matmul kernel against the 256-row kernels, whose bits it promises (one chain over K), and the oracle: rows and columns that
end inside a tile, fewer slabs than ring slots, more blocks of scales than their area holds, scale rows that are no whole number of
16-byte pieces or start at any byte; weights stored [N, K] and [K, N]."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as O
from tests.gpu_util import dev, hooked_library, hooks_lib

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _hooked():
    with hooked_library():
        yield


def _operands(rng, m, n, k, fmt):
    aq, asc = O.mx_quant(O.bf16_round(rng.standard_normal((m, k)).astype(np.float32)), fmt)
    bq, bsc = O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32)), fmt)
    # block scales over 2^16: with equal ones most sums are exact in any order
    return aq, (asc[:, :k // 32] + rng.integers(-16, 1, (m, k // 32))).astype(np.uint8), bq, (bsc[:, :k // 32] + rng.integers(-8, 9, (n, k // 32))).astype(np.uint8)


def _near(c, aq, asc, bq, bsc, fmt):
    """2-norm: products keep 2^-13 of the largest of eight (below 1e-3 on any sum of them), a bf16 output adds half a step of 2^-8."""
    gold = O.mx_dequant(aq, asc, fmt).astype(np.float32) @ O.mx_dequant(bq, bsc, fmt).astype(np.float32).T
    got = c.float().cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - gold) < 4e-3 * np.linalg.norm(gold)


@pytest.mark.parametrize("tm", [128, 192, 256])
@pytest.mark.parametrize("fmt,out,m,n,k", [("E4M3", "fp32", 1, 16, 128), ("E5M2", "fp32", 129, 132, 256), ("E4M3", "bf16", 260, 148, 640),
                                           ("E4M3", "fp32", 191, 300, 2176), ("E5M2", "fp16", 130, 264, 1024), ("E4M3", "fp32", 66, 20, 9344)])
def test_bits_of_the_256_row_kernels_on_both_weight_layouts(tm, fmt, out, m, n, k):
    from catccos_amd import ops
    rng = np.random.default_rng(m + n + k)
    aq, asc, bq, bsc = _operands(rng, m, n, k, fmt)
    a, a_s, b, b_s = dev(aq), dev(asc), dev(bq), dev(bsc)
    fb, fbs = O.to_file_layout(bq, bsc, True)
    h = hooks_lib()
    h.cmx_debug_force_tile(256, 256, 8)
    want = ops.mx_gemm(a, a_s, b, b_s, k, fmt, out)
    h.cmx_debug_force_tile(128, tm, 6)
    assert torch.equal(ops.mx_gemm(a, a_s, b, b_s, k, fmt, out), want)
    assert torch.equal(ops.mx_gemm_ex(a, a_s, dev(fb), dev(fbs), m, n, k, fmt, out, 0, 0), want)
    _near(want, aq, asc, bq, bsc, fmt)


@pytest.mark.parametrize("m,n,far", [(1100, 2048, "weights"), (128, 16448, "activations")])
def test_scale_rows_further_apart_than_32_bits_reach(m, n, far):
    """Default dispatch.  2048 weight rows of scales 4 MiB apart, 128 activation rows 64 MiB apart: byte offsets up to 2^33."""
    from catccos_amd import ops
    k, rng = 512, np.random.default_rng(m)
    aq, asc, bq, bsc = _operands(rng, m, n, k, "E4M3")
    a, a_s, b, b_s = dev(aq), dev(asc), dev(bq), dev(bsc)
    want = ops.mx_gemm(a, a_s, b, b_s, k, "E4M3", "fp32")
    near = b_s if far == "weights" else a_s
    apart = torch.empty((near.shape[0], 2 ** 33 // near.shape[0]), dtype=torch.uint8, device="cuda")[:, :near.shape[1]]
    apart.copy_(near)
    assert torch.equal(ops.mx_gemm(a, a_s if far == "weights" else apart, b, apart if far == "weights" else b_s, k, "E4M3", "fp32"), want)


@pytest.mark.parametrize("tm", [128, 192, 256])
@pytest.mark.parametrize("k", [384, 1152, 8832])
def test_scale_rows_at_any_byte(tm, k):
    """An odd pitch and an odd start; an output pitch wider than n keeps its rest."""
    from catccos_amd import _lib, ops
    rng = np.random.default_rng(k)
    m, n, pitch = 70, 45, k // 32 | 1
    aq, asc, bq, bsc = _operands(rng, m, n, k, "E4M3")
    a, b = dev(aq), dev(bq)
    hooks_lib().cmx_debug_force_tile(128, tm, 6)
    want = ops.mx_gemm(a, dev(asc), b, dev(bsc), k, "E4M3", "fp32")

    def shifted(s):
        buf = torch.full((1 + s.shape[0] * pitch,), 200, dtype=torch.uint8, device="cuda")
        buf[1:].view(s.shape[0], pitch)[:, :k // 32] = dev(s)
        return buf[1:]
    sa, sb, got = shifted(asc), shifted(bsc), torch.full((m, n + 3), 7.0, device="cuda")
    _lib.check(_lib.load().cmx_mx_gemm(a.data_ptr(), k, sa.data_ptr(), pitch, b.data_ptr(), k, sb.data_ptr(), pitch, got.data_ptr(), n + 3, m, n, k,
                                       ops.FMT["E4M3"], ops.OUT["fp32"], torch.cuda.current_stream().cuda_stream))
    assert torch.equal(got[:, :n], want) and bool((got[:, n:] == 7.0).all())


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("fmt,m,n,k", [("E4M3", 1, 16, 128), ("E5M2", 17, 68, 1152), ("E4M3", 65, 140, 2176), ("E4M3", 300, 1076, 640), ("E4M3", 280, 4100, 256),
                                       ("E4M3", 37, 64, 10496)])
def test_split_k_on_k_slow_weights_gives_the_bits_of_k_contiguous_ones(waves, fmt, m, n, k):
    """Tiles of 64 columns x 16, 32 (300 x 1076) and 64 rows (280 x 4100, four wavefronts); more scales than are in flight together."""
    from catccos_amd import ops
    rng = np.random.default_rng(m + n + k)
    aq, asc, bq, bsc = _operands(rng, m, n, k, fmt)
    a, a_s = dev(aq), dev(asc)
    fb, fbs = O.to_file_layout(bq, bsc, True)
    hooks_lib().cmx_debug_force_ksplit(4, 4, waves)
    want = ops.mx_gemm(a, a_s, dev(bq), dev(bsc), k, fmt, "fp32")
    assert torch.equal(ops.mx_gemm_ex(a, a_s, dev(fb), dev(fbs), m, n, k, fmt, "fp32", 0, 0), want)
    _near(want, aq, asc, bq, bsc, fmt)


@pytest.mark.parametrize("m,n,k", [(33, 3008, 512), (5, 512, 4224), (400, 2500, 1024), (700, 3008, 512), (1030, 4100, 640), (1300, 4096, 1024), (1700, 4092, 512), (1700, 4090, 512), (700, 3008, 576)])
def test_chosen_kernels_give_one_result_for_both_weight_layouts(m, n, k):
    """Sizes of the split-K tiles and of one round of each ring tile, and beside them what has the weights rewritten: columns no multiple of four, K no whole
    number of slabs."""
    from catccos_amd import ops
    rng = np.random.default_rng(m + n + k)
    aq, asc, bq, bsc = _operands(rng, m, n, k, "E4M3")
    fb, fbs = O.to_file_layout(bq, bsc, True)
    want = ops.mx_gemm(dev(aq), dev(asc), dev(bq), dev(bsc), k)
    assert torch.equal(ops.mx_gemm_ex(dev(aq), dev(asc), dev(fb), dev(fbs), m, n, k, trans_b=0), want)
    _near(want, aq, asc, bq, bsc, "E4M3")


@pytest.mark.parametrize("tile", [(128, 128), (128, 256), (256, 128)])
@pytest.mark.parametrize("counts,n,k", [([1, 0, 127, 128, 129, 0, 257, 66], 320, 512), ([300, 2], 192, 1152), ([0, 5, 0], 64, 128)])
def test_grouped_problems_give_the_bits_of_the_256_row_kernels(tile, counts, n, k):
    """Groups that end at and beside a tile's last row, empty ones, gate and up halves that end inside a tile."""
    from catccos_amd import ops
    rng = np.random.default_rng(sum(counts) + n)
    m, e = sum(counts), len(counts)
    aq, asc, bq, bsc = _operands(rng, m, e * n, k, "E4M3")
    a, a_s, w, w_s, cnt = dev(aq), dev(asc), dev(bq.reshape(e, n, k)), dev(bsc.reshape(e, n, -1)), dev(np.array(counts, dtype=np.int32))
    h = hooks_lib()

    def outputs():
        c = torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.mx_gmm(a, a_s, w, w_s, cnt, k, c=c)
        return [*ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k, want_bf16=True), *ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k)[:2],
                ops.mx_gmm(a, a_s, w, w_s, cnt, k, "E5M2", "fp32"), c]
    h.cmx_debug_force_tile(256, 256, 8)
    want = outputs()
    h.cmx_debug_force_tile(*tile, 6)
    for got, ref in zip(outputs(), want):
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8))
    assert bool((want[-1][m:].float() == 7.0).all())


@pytest.mark.parametrize("m,n,k", [(100, 1024, 3328), (100, 1024, 3456), (100, 768, 4096), (65, 2560, 8192), (300, 2816, 8192), (300, 2752, 8192), (600, 2368, 7168)])
def test_both_sides_of_the_k_slow_lines(m, n, k):
    """Default dispatch of split-K problems, weights read as they lie or behind the pass: the bits of K-contiguous weights."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    codes = lambda *shape: torch.randint(0, 0x70, shape, dtype=torch.uint8, device="cuda", generator=g)
    scales = lambda *shape: torch.randint(110, 125, shape, dtype=torch.uint8, device="cuda", generator=g)
    a, a_s, b, b_s = codes(m, k), scales(m, k // 32), codes(n, k), scales(n, k // 32)
    got = ops.mx_gemm_ex(a, a_s, b.t().contiguous(), b_s.view(n, k // 64, 2).permute(1, 0, 2).contiguous(), m, n, k, "E4M3", "fp32", trans_b=0)
    assert torch.equal(got, ops.mx_gemm(a, a_s, b, b_s, k, "E4M3", "fp32"))


@pytest.mark.parametrize("experts,avg,n,k", [(8, 100, 1024, 1024), (16, 100, 2048, 3072), (8, 200, 2048, 1024), (16, 100, 2048, 1024)])
def test_chosen_grouped_kernels(experts, avg, n, k):
    """Averages that take each of the ring tiles, and one that stays: the bits of the 256-row kernel either way."""
    from catccos_amd import ops
    rng = np.random.default_rng(avg)
    counts = rng.multinomial(experts * avg, np.full(experts, 1 / experts)).astype(np.int32)
    m = int(counts.sum())
    aq, asc, bq, bsc = _operands(rng, m, 256, k, "E4M3")
    w, w_s = dev(np.resize(bq, (experts, n, k))), dev(np.resize(bsc, (experts, n, k // 32)))
    a, a_s, cnt = dev(aq), dev(asc), dev(counts)

    def outputs():
        return [*ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k)[:2], ops.mx_gmm(a, a_s, w, w_s, cnt, k)]
    chosen = outputs()
    hooks_lib().cmx_debug_force_tile(256, 256, 8)
    for got, ref in zip(chosen, outputs()):
        assert torch.equal(got, ref)


@pytest.mark.parametrize("tile", [(128, 128), (128, 256), (256, 128)])
@pytest.mark.parametrize("out", ["fp32", "bf16"])
@pytest.mark.parametrize("counts,n,k", [([1, 0, 127, 128, 129, 0, 257, 66], 320, 512), ([300, 2], 196, 1280), ([0, 5, 0], 64, 256), ([70], 130, 17664)])
def test_grouped_fp4_gives_the_bits_of_the_256_row_kernel(tile, out, counts, n, k):
    """Two dwords of scales a slab: a last piece of them in part (1280), more than their area holds (17664), less than a piece (256)."""
    from catccos_amd import ops
    rng = np.random.default_rng(sum(counts) + k)
    m, e = sum(counts), len(counts)
    aq, asc, bq, bsc = _operands(rng, m, e * n, k, "E2M1")
    a, w = dev(O.pack_fp4(aq)), dev(O.pack_fp4(bq).reshape(e, n, k // 2))
    args = (a, dev(asc), w, dev(bsc.reshape(e, n, -1)), dev(np.array(counts, dtype=np.int32)), k, "E2M1", out)
    h = hooks_lib()
    h.cmx_debug_force_tile(256, 256, 8)
    want = ops.mx_gmm(*args)
    h.cmx_debug_force_tile(*tile, 6)
    assert torch.equal(ops.mx_gmm(*args), want)


@pytest.mark.parametrize("tile", [(128, 128), (128, 256), (256, 128)])
@pytest.mark.parametrize("out", ["fp32", "bf16"])
@pytest.mark.parametrize("counts,n,k", [([1, 0, 127, 128, 129, 0, 257, 66], 320, 512), ([300, 2], 192, 128), ([0, 5, 0], 64, 1152)])
def test_grouped_int8_gives_the_bits_of_the_256_row_kernel(tile, out, counts, n, k):
    """Whole-number sums and the same arithmetic behind them; fewer slabs than ring slots."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    m, e = sum(counts), len(counts)
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (e, n, k), dtype=torch.int8, device="cuda", generator=g)
    channel, token = torch.rand(e * n, device="cuda", generator=g) * 1e-4, torch.rand(m, device="cuda", generator=g)
    args = (a, token, w, channel, dev(np.array(counts, dtype=np.int32)), n, k, 1, out)
    h = hooks_lib()
    h.cmx_debug_force_tile(256, 256, 8)
    want = ops.int8_gmm_dequant_swiglu(*args)
    h.cmx_debug_force_tile(*tile, 6)
    assert torch.equal(ops.int8_gmm_dequant_swiglu(*args), want)


@pytest.mark.parametrize("counts,rows,n,k", [
    # by the sizes (most tiles of two rounds), and by the launch that fills the tables; the 256 x 128 side, and the 256 x 256 one
    ([90] * 12, 1080, 4096, 512),                                      # sizes, one round of either: 256 x 128
    ([1300, 0, 0, 90] + [3] * 8, 1414, 4096, 512),                     # sizes, two rounds against one: 256 x 256
    ([100, 130, 140] * 5, 1850, 4096, 2048),                           # K >= 2048, groups of a little more than 128 rows: 256 x 256
    ([90] * 40, 3600, 4096, 512),                                      # tables, three rounds of either: 256 x 128
    ([2000, 1500] + [0] * 38, 3500, 4096, 512),                        # tables, two rounds against one: 256 x 256
    ([60, 70, 129, 5] * 75, 19800, 1024, 512),                         # tables of more groups than a scan takes: 256 x 128
    ([9000, 0, 7000] + [1] * 298, 16298, 1024, 512),                   # the same, 256 x 256
    ([2 ** 31 - 1, -4] + [9] * 8, 1200, 4096, 512),                    # sizes past the rows that there are, negative ones
    ([2 ** 31 - 1, -4, 7, 2 ** 31 - 1] + [9] * 16, 1900, 4096, 512),   # the same in tables
    ([1100, 0, 64, 65, 1, 800, 33, 200] + [0] * 52, 2263, 4096, 512),  # small groups to split-K, the choice for the others
    ([110] * 20, 2200, 4096, 384),                                     # K < 512: 256 x 256 tiles without a choice
    ([60, 70, 129, 5] * 75, 19800, 128, 512)])                         # n <= 128: 128 x 128 tiles of more than a round
def test_chosen_int8_kernels(counts, rows, n, k):
    """Whatever of the 256 x 128 and 256 x 256 tiles the host or the device takes: one result, that of the 256-row kernel alone."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    e = len(counts)
    a = torch.randint(-127, 128, (rows, k), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-127, 128, (e, n, k), dtype=torch.int8, device="cuda", generator=g)
    channel, token = torch.rand(e * n, device="cuda", generator=g) * 1e-4, torch.rand(rows, device="cuda", generator=g)
    args = (a, token, w, channel, dev(np.array(counts, dtype=np.int32)), n, k, 1)
    chosen = ops.int8_gmm_dequant_swiglu(*args)
    hooks_lib().cmx_debug_force_ksplit(-1, 0, 0)
    hooks_lib().cmx_debug_force_tile(256, 256, 8)
    assert torch.equal(ops.int8_gmm_dequant_swiglu(*args), chosen) and chosen.abs().max() > 0


@pytest.mark.parametrize("kind,k", [("E4M3", 512), ("E2M1", 512), ("SwiGLU", 3072), ("SwiGLU", 512)])
@pytest.mark.parametrize("n", [64, 128, 192])
def test_narrow_weights_in_many_groups(kind, k, n):
    """More than a round of 128 x 128 tiles, which n <= 128 takes and 192 does not: the bits of the 256-row kernel."""
    from catccos_amd import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    counts = torch.tensor([70, 0, 129, 128] * 60, dtype=torch.int32, device="cuda")
    e, m, kb = len(counts), int(counts.sum()), k // 2 if kind == "E2M1" else k
    codes = lambda *shape: torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xF7
    scales = lambda *shape: torch.randint(110, 125, shape, dtype=torch.uint8, device="cuda", generator=g)
    args = (codes(m, kb), scales(m, k // 32), codes(e, n, kb), scales(e, n, k // 32), counts, k)
    call = (lambda: ops.mx_gmm_swiglu_quant(*args)[:2]) if kind == "SwiGLU" else (lambda: [ops.mx_gmm(*args, kind)])
    chosen = call()
    hooks_lib().cmx_debug_force_tile(256, 256, 8)
    for got, ref in zip(chosen, call()):
        assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8)) and bool((ref != 0).any())


@pytest.mark.parametrize("kernel", ["ring", "split-K", "INT8"])
@pytest.mark.parametrize("sizes,rows", [([5, -3, 0, 70, 1], 76), ([40, 2 ** 31 - 1, 2 ** 31 - 1, 9], 300), ([0, 0, 0], 10), ([1] * 256, 256),
                                        ([3, 0, 66, 1] * 64, 4300), ([2 ** 31 - 1] * 256, 130)])
def test_tiles_located_by_sizes_are_those_of_the_tables(kernel, sizes, rows):
    """Up to 256 groups a launch reads the sizes themselves, more go through tables: empty groups behind the last one change
    nothing.  Negative sizes count as zero, rows past the operand are cut off."""
    from catccos_amd import ops
    rng = np.random.default_rng(rows)
    n, k, many = 64, 512, 300
    aq, asc, bq, bsc = _operands(rng, rows, 4 * n, k, "E4M3")
    a, a_s, w, w_s = dev(aq), dev(asc), dev(np.resize(bq, (many, n, k))), dev(np.resize(bsc, (many, n, k // 32)))
    h = hooks_lib()
    if kernel == "ring":
        h.cmx_debug_force_tile(128, 128, 6)
    else:
        h.cmx_debug_force_ksplit(4, 4, 4)

    def outputs(counts):
        e = len(counts)
        cnt = dev(np.array(counts, dtype=np.int32))
        c = torch.full((rows, n), 7.0, dtype=torch.bfloat16, device="cuda")
        if kernel == "INT8":
            out = torch.zeros((rows, n // 2), device="cuda")
            return ops.int8_gmm_dequant_swiglu(a.view(torch.int8), torch.ones(rows, device="cuda"), w[:e].view(torch.int8), torch.full((e * n,), 1e-5, device="cuda"),
                                               cnt, n, k, 1, c=out)
        return ops.mx_gmm(a, a_s, w[:e], w_s[:e], cnt, k, c=c)
    got, want = outputs(sizes), outputs(sizes + [0] * (many - len(sizes)))
    assert torch.equal(got, want)
    if kernel == "ring":
        done = min(sum(max(s, 0) for s in sizes), rows)
        assert bool((got[done:].float() == 7.0).all()) and not bool((got[:done].float() == 7.0).all(dim=1).any())


@pytest.mark.parametrize("tw,tm", [(128, 128), (256, 128), (128, 256)])
@pytest.mark.parametrize("want_bf16", [False, True])
def test_activation_codes_in_rows_of_four_byte_alignment(tw, tm, want_bf16):
    """A thread's eight codes leave in one store where rows start at eight bytes, else in two; what lies between the rows is left alone."""
    from catccos_amd import ops
    counts, n, k = [130, 0, 257, 3], 320, 640
    m, g = sum(counts) + 2, torch.Generator(device="cuda")
    g.manual_seed(tw + tm)
    codes = lambda *shape: torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0x77
    scales = lambda *shape: torch.randint(112, 124, shape, dtype=torch.uint8, device="cuda", generator=g)
    a, a_s, w, w_s = codes(m, k), scales(m, k // 32), codes(len(counts), n, k), scales(len(counts), n, k // 32)
    cnt = dev(np.array(counts, dtype=np.int32))
    hooks_lib().cmx_debug_force_tile(tw, tm, 6)

    def outputs(pad, start):
        """codes in rows of n / 2 + pad bytes, the first row `start` bytes behind a multiple of 16"""
        buf = torch.full((m * (n // 2 + pad) + 16,), 0x55, dtype=torch.uint8, device="cuda")
        rows = buf[start:start + m * (n // 2 + pad)].view(m, -1)
        s = torch.full((m, ops.scale_cols(n // 2)), 0x55, dtype=torch.uint8, device="cuda")
        act = ops.mx_gmm_swiglu_quant(a, a_s, w, w_s, cnt, k, want_bf16=want_bf16, outs=(rows[:, :n // 2], s))[2]
        assert bool((rows[:, n // 2:] == 0x55).all()) and bool((buf[:start] == 0x55).all()) and bool((buf[start + rows.numel():] == 0x55).all())
        return [rows[:, :n // 2], s] + ([act] if want_bf16 else [])
    want = outputs(0, 0)
    assert bool((want[0][:m - 2] != 0x55).any(dim=1).all()) and bool((want[0][m - 2:] == 0x55).all())
    for pad, start in (4, 0), (8, 4), (0, 4):
        for x, y in zip(outputs(pad, start), want):
            assert torch.equal(x, y)
