"""The split-K matmul kernels (few activation rows or few tiles) against the oracle, at the edges of their tiles: one row, a row
past a fragment, a partly filled slab of K, columns that end inside a tile, and every epilogue; row-major and pre-tiled weights
give the same bits."""
import numpy as np
import pytest
import torch

from oracle import int8_oracle as Q
from oracle import mx_oracle as O
from tests.gpu_util import dev, host, close_bf16, hooked_library, hooks_lib

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 8), (1, 2, 8), (2, 1, 8), (2, 2, 8), (2, 4, 8), (4, 1, 8), (4, 2, 8), (4, 4, 8), (4, 4, 4)]


@pytest.fixture(autouse=True)
def _hooked():
    with hooked_library():
        yield


def _mx(rng, rows, k, fmt, std=1.0):
    return O.mx_quant(O.bf16_round(rng.standard_normal((rows, k)).astype(np.float32) * std), fmt)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("fmt,m,n,k", [("E4M3", 1, 8, 32), ("E5M2", 17, 40, 96), ("E4M3", 65, 136, 1216), ("E4M3", 64, 72, 2304),
                                       ("E2M1", 33, 130, 160), ("E2M1", 64, 64, 2560)])
def test_dense_tiles(shape, fmt, m, n, k):
    """fp32 outputs: the matrix cores align eight consecutive 8-bit products to the largest of them and drop what lies below 2^-13
    of it (so 1e-3 relative and, near zero, 1e-2 on sums whose terms are of order ten); FP4 products are short enough to be
    exact, which leaves the order of the fp32 additions."""
    from catccos_amd import ops
    hooks_lib().cmx_debug_force_ksplit(*shape)
    rng = np.random.default_rng(m + n + k)
    aq, asc = _mx(rng, m, k, fmt)
    bq, bsc = _mx(rng, n, k, fmt)
    pack = O.pack_fp4 if fmt == "E2M1" else (lambda x: x)
    gold = O.mx_dequant(aq, asc, fmt).astype(np.float64) @ O.mx_dequant(bq, bsc, fmt).astype(np.float64).T
    c = host(ops.mx_gemm(dev(pack(aq)), dev(asc), dev(pack(bq)), dev(bsc), k, fmt, "fp32"))
    rtol, atol = (1e-5, 1e-4) if fmt == "E2M1" else (1e-3, 1e-2)
    assert np.allclose(c, gold, rtol=rtol, atol=atol), np.abs(c - gold).max()
    bad, worst = close_bf16(host(ops.mx_gemm(dev(pack(aq)), dev(asc), dev(pack(bq)), dev(bsc), k, fmt, "bf16")), gold)
    assert bad == 0, (bad, worst)


# the last K of a ring of two and of four slots, the first of the next, a slab in part behind either
@pytest.mark.parametrize("shape", [(1, 1, 8), (1, 2, 8), (2, 1, 8), (2, 2, 8)])
@pytest.mark.parametrize("fmt,k", [("E4M3", 2048), ("E4M3", 2080), ("E5M2", 2176), ("E4M3", 4096), ("E4M3", 4128), ("E4M3", 4224), ("E2M1", 4096), ("E2M1", 4352),
                                   ("E2M1", 8192), ("E2M1", 8448)])
def test_rings_of_every_length(shape, fmt, k):
    """Against the 64 x 64 tile, whose ring has one length: eight partial sums on either, so the same bits."""
    from catccos_amd import ops
    rng = np.random.default_rng(k)
    m, n = 21, 40
    aq, asc = _mx(rng, m, k, fmt)
    bq, bsc = _mx(rng, n, k, fmt)
    pack = O.pack_fp4 if fmt == "E2M1" else (lambda x: x)
    args = dev(pack(aq)), dev(asc), dev(pack(bq)), dev(bsc), k, fmt, "fp32"
    hooks_lib().cmx_debug_force_ksplit(4, 4, 8)
    want = host(ops.mx_gemm(*args))
    hooks_lib().cmx_debug_force_ksplit(*shape)
    assert np.array_equal(host(ops.mx_gemm(*args)), want) and np.abs(want).max() > 0


def test_scale_rows_that_are_not_dword_aligned_and_an_output_pitch():
    """K = 96: three scales a row, fewer than the dword that longer rows end in, at a pitch of 5.  Output rows wider than n: the rest
    keeps its poison."""
    from catccos_amd import _lib
    rng = np.random.default_rng(4)
    m, n, k, ldc = 19, 21, 96, 24
    aq, asc = _mx(rng, m, k, "E4M3")
    bq, bsc = _mx(rng, n, k, "E4M3")
    a_s, b_s = dev(np.pad(asc, ((0, 0), (0, 1)))), dev(np.pad(bsc, ((0, 0), (0, 1))))
    c = torch.full((m, ldc), 7.0, dtype=torch.bfloat16, device="cuda")
    lib = _lib.load()
    a, b = dev(aq), dev(bq)
    _lib.check(lib.cmx_mx_gemm(a.data_ptr(), k, a_s.data_ptr(), 5, b.data_ptr(), k, b_s.data_ptr(), 5, c.data_ptr(), ldc, m, n, k, 0, 0,
                               torch.cuda.current_stream().cuda_stream))
    gold = O.mx_dequant(aq, asc).astype(np.float64) @ O.mx_dequant(bq, bsc).astype(np.float64).T
    bad, worst = close_bf16(host(c)[:, :n], gold)
    assert bad == 0, (bad, worst)
    assert bool((c[:, n:].float() == 7.0).all())


COUNTS = [[1, 0, 16, 17, 33, 0, 64, 65, 2], [0, 0, 3], [130, 1]]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("n,k", [(320, 512), (192, 1536)])
def test_grouped_swiglu_and_store_on_both_weight_layouts(counts, n, k):
    from catccos_amd import ops
    hooks_lib().cmx_debug_force_ksplit(4, 4, 4)
    rng = np.random.default_rng(sum(counts) + n)
    m = sum(counts)
    aq, asc = _mx(rng, m, k, "E4M3")
    w = [O.mx_quant(O.bf16_round(rng.standard_normal((n, k)).astype(np.float32) / np.sqrt(k)), "E4M3", "lut") for _ in counts]
    wq, ws = np.stack([a for a, _ in w]), np.stack([b for _, b in w])
    a, a_s, wd, wsd, cnt = dev(aq), dev(asc), dev(wq), dev(ws), dev(np.array(counts, dtype=np.int32))
    codes, scales, act = ops.mx_gmm_swiglu_quant(a, a_s, wd, wsd, cnt, k, want_bf16=True)
    bad, worst = close_bf16(host(act), O.bf16_bits_to_f32(O.gmm1_swiglu_quant(aq, asc, wq, ws, counts)[1]), rtol=2e-2)
    assert bad == 0, (bad, worst)
    q2, s2 = O.mx_quant_bf16(host(act), "E4M3", "rne")
    assert np.array_equal(host(codes), q2) and np.array_equal(host(scales), s2)
    for weights in (wd, ops.pretile_weights(wd, True)):
        c, s, _ = ops.mx_gmm_swiglu_quant(a, a_s, weights, wsd, cnt, k)
        assert torch.equal(c, codes) and torch.equal(s, scales)
    y = torch.full((m + 2, n), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.mx_gmm(a, a_s, wd, wsd, cnt, k, c=y)
    bad, worst = close_bf16(host(y)[:m], O.mx_gmm_f32(aq, asc, wq, ws, counts))
    assert bad == 0 and bool((y[m:].float() == 7.0).all()), (bad, worst)
    assert torch.equal(y[:m], ops.mx_gmm(a, a_s, ops.pretile_weights(wd, False), wsd, cnt, k))


@pytest.mark.parametrize("counts", COUNTS)
def test_grouped_fp4(counts):
    from catccos_amd import ops
    hooks_lib().cmx_debug_force_ksplit(4, 4, 4)
    rng = np.random.default_rng(sum(counts))
    n, k, m = 200, 800, sum(counts)
    aq, asc = O.mx_quant(rng.uniform(-2, 2, (m, k)).astype(np.float32), "E2M1")
    w = [O.mx_quant(rng.uniform(-2, 2, (n, k)).astype(np.float32), "E2M1") for _ in counts]
    wq, ws = np.stack([a for a, _ in w]), np.stack([b for _, b in w])
    c = ops.mx_gmm(dev(O.pack_fp4(aq)), dev(asc), dev(O.pack_fp4(wq)), dev(ws), dev(np.array(counts, dtype=np.int32)), k, "E2M1", "fp32")
    gold = O.mx_gmm_f32(aq, asc, wq, ws, counts, "E2M1", "E2M1")
    assert np.allclose(host(c), gold, rtol=1e-5, atol=1e-4)


def test_dense_tiles_refuse_groups():
    """The kernels of dense problems have no code that looks for groups: a grouped problem on one of their tiles is an error of the host."""
    from catccos_amd import _lib, ops
    hooks_lib().cmx_debug_force_ksplit(1, 1, 8)
    u8 = lambda *shape: torch.zeros(shape, dtype=torch.uint8, device="cuda")
    with pytest.raises(_lib.CmxError, match="64 x 64 only"):
        ops.mx_gmm(u8(32, 128), u8(32, 4), u8(2, 64, 128), u8(2, 64, 4), torch.tensor([16, 16], dtype=torch.int32, device="cuda"), 128)


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("out", ["fp32", "bf16"])
def test_grouped_int8(counts, out):
    from catccos_amd import ops
    hooks_lib().cmx_debug_force_ksplit(4, 4, 4)
    rng = np.random.default_rng(sum(counts) + 1)
    n, k, m, e = 192, 640, sum(counts), len(counts)
    a = rng.integers(-128, 128, size=(m, k), dtype=np.int8)
    b = rng.integers(-128, 128, size=(e, k, n), dtype=np.int8)
    ch = Q.truncate_scale(rng.standard_normal(e * n).astype(np.float32) * 1e-4)
    ts = (np.abs(rng.standard_normal(m)) / 127 + 1e-3).astype(np.float32)
    args = (dev(a), dev(ts), dev(np.ascontiguousarray(b.transpose(0, 2, 1))), dev(ch), dev(np.array(counts, dtype=np.int32)), n, k, 1, out)
    got = ops.int8_gmm_dequant_swiglu(*args)
    # whole-number sums and the same arithmetic behind them: the bits of the 256-row kernel
    hooks_lib().cmx_debug_force_ksplit(0, 0, 0)
    hooks_lib().cmx_debug_force_tile(256, 256, 8)
    assert torch.equal(got, ops.int8_gmm_dequant_swiglu(*args))
    # and the oracle's: INT32 sums and the fp16 step are exact, the sigmoid is within a few ulp
    gold = Q.gmm_dequant_swiglu(a, ts, b, ch, counts)
    assert np.allclose(got.float().cpu().numpy(), gold, rtol=1e-5 if out == "fp32" else 1e-2, atol=1e-7 if out == "fp32" else 1e-3)


@pytest.mark.parametrize("shape", [(1, 1, 8), (4, 4, 8), (4, 4, 4)])
@pytest.mark.parametrize("fmt,k", [("E4M3", 1952), ("E4M3", 8736), ("E2M1", 1952), ("E5M2", 496 * 32)])
def test_scale_rows_at_any_byte_give_the_bits_of_aligned_ones(shape, fmt, k):
    """61 scales (three 16-byte pieces and a tail of 13 bytes), 273 (more pieces than are in flight together, a tail of one)
    and 496 (whole pieces) in rows of an odd pitch that start at an odd address: the result of the same scales in aligned
    rows, and the oracle's."""
    from catccos_amd import _lib, ops
    hooks_lib().cmx_debug_force_ksplit(*shape)
    rng = np.random.default_rng(k)
    m, n, nb = 37, 45, k // 32
    aq, asc = _mx(rng, m, k, fmt)
    bq, bsc = _mx(rng, n, k, fmt)
    pack = O.pack_fp4 if fmt == "E2M1" else (lambda x: x)
    a, b, pitch = dev(pack(aq)), dev(pack(bq)), nb | 1
    want = ops.mx_gemm(a, dev(asc), b, dev(bsc), k, fmt, "fp32")

    def shifted(s):
        buf = torch.full((1 + s.shape[0] * pitch,), 200, dtype=torch.uint8, device="cuda")
        buf[1:].view(s.shape[0], pitch)[:, :nb] = dev(s)[:, :nb]
        return buf[1:]
    sa, sb, got = shifted(asc), shifted(bsc), torch.empty_like(want)
    lib = _lib.load()
    _lib.check(lib.cmx_mx_gemm(a.data_ptr(), a.shape[1], sa.data_ptr(), pitch, b.data_ptr(), b.shape[1], sb.data_ptr(), pitch, got.data_ptr(),
                               n, m, n, k, ops.FMT[fmt], ops.OUT["fp32"], torch.cuda.current_stream().cuda_stream))
    assert torch.equal(got, want)
    gold = O.mx_dequant(aq, asc, fmt).astype(np.float64) @ O.mx_dequant(bq, bsc, fmt).astype(np.float64).T
    bad, worst = close_bf16(host(got.to(torch.bfloat16)), gold)
    assert bad == 0, (bad, worst)


@pytest.mark.parametrize("fmt,out,m,n,k", [("E4M3", "bf16", *mnk) for mnk in ((1000, 4000, 512), (1024, 4104, 512), (1024, 4096, 2048), (1024, 4096, 2176),
                                                                               (2048, 4096, 96), (2049, 4096, 96), (520, 4000, 256))] +
                         [("E5M2", "bf16", 1000, 4000, 512), ("E4M3", "fp16", 1000, 4000, 512), ("E5M2", "fp32", 1000, 4004, 512),
                          ("E4M3", "fp32", 2100, 4104, 512), ("E4M3", "bf16", 2100, 4104, 1024), ("E2M1", "fp32", 2100, 4104, 512), ("E2M1", "bf16", 1000, 4104, 1024)])
@pytest.mark.parametrize("aligned", [True, False])
def test_sizes_on_both_sides_of_the_dense_rules(fmt, out, m, n, k, aligned):
    """256 and more 128 x 128 tiles; more than 1024 64 x 64 tiles, 2048 where K is no whole number of slabs; the kernel that the
    library chooses against the oracle.  Scale rows at an odd pitch (which takes the 128 x 128 and 256-row tiles to the
    register-staged kernel) give the bits of aligned ones."""
    from catccos_amd import _lib, ops
    rng = np.random.default_rng(m + n + k)
    aq, asc = _mx(rng, m, k, fmt)
    bq, bsc = _mx(rng, n, k, fmt)
    pack = O.pack_fp4 if fmt == "E2M1" else (lambda x: x)
    a, b = dev(pack(aq)), dev(pack(bq))
    if not aligned:
        asc = (asc + rng.integers(-8, 9, asc.shape)).astype(np.uint8)      # (with equal scales most sums are exact in any order)
    c = ops.mx_gemm(a, dev(asc), b, dev(bsc), k, fmt, out)
    if not aligned:
        pitch = (k // 32) | 1
        sa, sb = dev(np.pad(asc[:, :k // 32], ((0, 0), (0, pitch - k // 32)))), dev(np.pad(bsc[:, :k // 32], ((0, 0), (0, pitch - k // 32))))
        got = torch.empty_like(c)
        _lib.check(_lib.load().cmx_mx_gemm(a.data_ptr(), a.shape[1], sa.data_ptr(), pitch, b.data_ptr(), b.shape[1], sb.data_ptr(), pitch, got.data_ptr(), n, m, n,
                                           k, ops.FMT[fmt], ops.OUT[out], torch.cuda.current_stream().cuda_stream))
        assert torch.equal(got, c)
        return
    gold = (O.mx_dequant(aq, asc, fmt).astype(np.float32) @ O.mx_dequant(bq, bsc, fmt).astype(np.float32).T)
    if out == "bf16":
        bad, worst = close_bf16(host(c), gold)
        assert bad == 0, (bad, worst)
    else:
        # products as in test_dense_tiles; fp16 adds half a step
        assert np.allclose(host(c).astype(np.float64), gold, rtol=1e-3 + 2.0 ** -11, atol=1e-2 + 2.0 ** -11)


@pytest.mark.parametrize("kernel", ["split-K", "256-row"])
@pytest.mark.parametrize("p0,p1", [(0, 5), (0, 20), (9, 70), (40, 127)])
def test_eight_consecutive_products_are_aligned_to_the_largest(kernel, p0, p1):
    """What the tolerances of the 8-bit matmuls rest on, for both instruction shapes (16 x 16 x 128, 32 x 32 x 64): row r is 2^8 at
    p0, -2^8 at p1 and s at r against weights of one.  s = 2^-5 always arrives; s = 2^-6, less than 2^-13 of the largest product,
    is lost beside p0 or p1 among the same eight, and only there."""
    from catccos_amd import ops
    if kernel == "split-K":
        hooks_lib().cmx_debug_force_ksplit(1, 1, 8)
    else:
        hooks_lib().cmx_debug_force_tile(256, 256, 8)
    k = 128
    r = np.array([i for i in range(k) if i not in (p0, p1)])
    b, bs = dev(np.full((16, k), 0x38, dtype=np.uint8)), dev(np.full((16, 4), 127, dtype=np.uint8))
    for code, s in ((0x10, 2.0 ** -5), (0x08, 2.0 ** -6)):
        a = np.zeros((len(r), k), dtype=np.uint8)
        a[:, p0], a[:, p1] = 0x78, 0xF8
        a[np.arange(len(r)), r] = code
        c = host(ops.mx_gemm(dev(a), dev(np.full((len(r), 4), 127, dtype=np.uint8)), b, bs, k, "E4M3", "fp32"))
        kept = (s > 2.0 ** -6) | ((r // 8 != p0 // 8) & (r // 8 != p1 // 8))
        assert np.array_equal(c, np.where(kept, s, 0.0)[:, None].repeat(16, 1).astype(np.float32))


SKEWED = [1300, 0, 64, 65, 1, 700, 33, 63] + [0] * 55 + [66]


@pytest.mark.parametrize("cut", [0, 5])
def test_skewed_groups_take_the_kernel_of_their_size(cut):
    """64 groups that average 36 rows, 1152 tiles of 64 x 64 where 1024 are the most for one launch: the groups of at most 64 rows have the bits of the split-K
    kernel (four partial sums), the others those of the 256-row kernel (one chain over K), on row-major and on pre-tiled
    weights.  cut: the operands hold five rows less than the groups ask for, which makes the last group one of 61."""
    from catccos_amd import _lib, ops
    h = hooks_lib()
    rng = np.random.default_rng(11 + cut)
    n, k, e = 2048, 512, len(SKEWED)
    m = sum(SKEWED) - cut
    counts = SKEWED[:-1] + [SKEWED[-1] - cut]
    small = np.repeat([0 < c <= 64 for c in counts], counts)
    small = torch.from_numpy(small).cuda()
    aq, asc = _mx(rng, m, k, "E4M3")
    wq, ws = _mx(rng, e * n, k, "E4M3", 1 / np.sqrt(k))
    # block scales over 2^16: with equal ones the sums are short enough to be exact in any order
    asc = (asc + rng.integers(-8, 9, asc.shape)).astype(np.uint8)
    wq, ws = wq.reshape(e, n, k), ws.reshape(e, n, -1)
    a, a_s, w, w_s, cnt = dev(aq), dev(asc), dev(wq), dev(ws), dev(np.array(SKEWED, dtype=np.int32))

    def store(weights=w, out="fp32"):
        return ops.mx_gmm(a, a_s, weights, w_s, cnt, k, "E4M3", out)

    def swiglu(weights=w):
        return torch.cat(ops.mx_gmm_swiglu_quant(a, a_s, weights, w_s, cnt, k)[:2], dim=1)

    ai = torch.randint(-127, 128, (m, k), dtype=torch.int8, device="cuda")
    wi = torch.randint(-127, 128, (e, n, k), dtype=torch.int8, device="cuda")
    channel, token = torch.rand(e * n, device="cuda") * 1e-3, torch.rand(m, device="cuda")

    def int8():
        return ops.int8_gmm_dequant_swiglu(ai, token, wi, channel, cnt, n, k, 1)

    calls = (store, swiglu, int8)
    chosen = [f() for f in calls]
    h.cmx_debug_force_ksplit(4, 4, 4)
    split = [f() for f in calls]
    h.cmx_debug_force_ksplit(0, 0, 0)
    h.cmx_debug_force_tile(256, 128, 5)
    chain = [f() for f in calls[:2]]
    h.cmx_debug_force_tile(0, 0, 0)
    assert float((split[0] != chain[0]).any(dim=1).float().mean()) > 0.9      # the two sides can be told apart
    for got, s, c in zip(chosen, split, chain):
        assert torch.equal(got[small], s[small])
        assert torch.equal(got[~small], c[~small])
    assert torch.equal(chosen[2], split[2])                                   # whole-number sums: the same on both
    assert torch.equal(swiglu(ops.pretile_weights(w, True)), chosen[1])
    assert torch.equal(store(ops.pretile_weights(w, False), "bf16"), store(out="bf16"))
    codes, scales = torch.zeros((m, n // 2), dtype=torch.uint8, device="cuda"), torch.zeros((m, n // 64), dtype=torch.uint8, device="cuda")
    _lib.check(h.cmx_mx_gmm_swiglu_quant_noalloc(a.data_ptr(), k, a_s.data_ptr(), a_s.shape[1], w.data_ptr(), w_s.data_ptr(), codes.data_ptr(),
                                                 n // 2, scales.data_ptr(), n // 64, None, cnt.data_ptr(), e, m, n, k,
                                                 torch.cuda.current_stream().cuda_stream))
    assert torch.equal(torch.cat((codes, scales), dim=1), chosen[1])
    gold = O.mx_gmm_f32(aq, asc, wq, ws, counts)
    assert np.linalg.norm(host(chosen[0]) - gold) < 1e-3 * np.linalg.norm(gold)       # products keep 2^-13 of the largest of eight
