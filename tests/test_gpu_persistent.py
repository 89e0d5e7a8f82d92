"""The persistent 256 x 256 kernels with 2 x 2 wavefronts: their walk through more and less than whole rounds of tiles.
Reference: the streaming kernel of the same tile, one tile per workgroup, whose K order is the
same, so the outputs are the same bits."""
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
