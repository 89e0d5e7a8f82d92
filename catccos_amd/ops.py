"""Thin torch-tensor front end of the C ABI (device memory and streams only).

Every function takes CUDA(=HIP) tensors, passes raw pointers to libcatccos_mx.so on
torch's current stream and returns tensors.  The calls of a layer allocate and call through _native_call; set-up and checking
functions through ctypes.  bf16 data may be given as
torch.bfloat16 or as int16/uint16 bit patterns.  No function here computes
anything in torch.
"""
from __future__ import annotations

from operator import index

import torch

from . import _lib


def _bind_native():
    """Puts the functions of the extension in the place of the two below, at the first call as for the library: what needs no kernel
    works without either."""
    global _run, _empty
    try:
        from . import _native_call
        if _native_call.torch_version != str(torch.__version__):
            raise ImportError(f"built for torch {_native_call.torch_version}, not {torch.__version__}")
    except ImportError as e:
        raise ImportError(f"catccos_amd/_native_call: {e}; build it with `python -m catccos_amd.build`") from e
    _run, _empty = _native_call.run, _native_call.empty


def _run(*args):
    _bind_native()
    return _run(*args)


def _empty(*args):
    _bind_native()
    return _empty(*args)


FMT = {"E4M3": 0, "E5M2": 1, "E2M1": 2, "E1M2": 3}
_FP4 = ("E2M1", "E1M2")
ROUND = {"rne": 0, "lut": 1}
OUT = {"bf16": 0, "fp16": 1, "fp32": 2}
_OUT_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


# not a public function of torch, so it may be missing
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_device = getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device


def _stream():
    # the handle of torch's current stream without a Stream object around it: 0.2 us of host time against 2.8, of 5 a call
    if _raw_stream is not None:
        return _raw_stream(_device())
    return torch.cuda.current_stream().cuda_stream


def _p(t: torch.Tensor):
    return t.data_ptr() if t is not None else None


def _launch(name, *args):
    """The entry point `name` on these tensors (GPU tensors, or ValueError), integers and Nones, and torch's current stream (...); a tuple (dtype,
    sizes) stands for a new tensor.  Returns the new tensors.  A whole number that the caller gives goes through index() first: as a tensor of one
    element it would be passed by its address."""
    out = _run(_lib.entries()[name], *args, ...)
    if out.__class__ is int:
        _lib.check(out)
    return out


def _brought(t):
    """Weights, an output or a workspace that the caller brings, for _run: these may also lie in pinned host memory, which kernels reach by
    its address (any other host tensor is passed on, and refused)."""
    return t if isinstance(t, torch.Tensor) and (t.is_cuda or not t.is_pinned()) else t.data_ptr()


def _no_new(*ts):
    """What a caller gives where _launch gets it as it is, and where a tuple would stand for a new tensor."""
    for t in ts:
        if isinstance(t, tuple):
            raise TypeError("expected a tensor, not a tuple")


def _need_cuda(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("expected a GPU tensor")


def scale_cols(cols: int) -> int:
    nb = (cols + 31) // 32
    return (nb + 1) // 2 * 2


def mx_quant(x: torch.Tensor, fmt: str = "E4M3", mode: str | None = None):
    """x: bf16 [rows, cols] -> (codes u8 [rows, cols or cols/2], scales u8 [rows, RoundUp2(cols/32)])."""
    assert x.dim() == 2 and x.element_size() == 2
    rows, cols = x.shape
    pitch, step = x.stride()
    assert step == 1
    fp4 = fmt in _FP4
    if mode is None:
        mode = "lut" if fp4 else "rne"
    ccols = (cols + 1) // 2 if fp4 else cols
    scols = scale_cols(cols)
    return _launch("cmx_mx_quant", x, pitch, (torch.uint8, rows, ccols), ccols, (torch.uint8, rows, scols), scols, rows, cols, FMT[fmt], ROUND[mode])


def mx_dequant(codes: torch.Tensor, scales: torch.Tensor, cols: int, fmt: str = "E4M3") -> torch.Tensor:
    _need_cuda(codes, scales)
    rows = codes.shape[0]
    out = torch.empty((rows, cols), dtype=torch.float32, device=codes.device)
    lib = _lib.load()
    _lib.check(lib.cmx_mx_dequant(_p(codes), codes.stride(0), _p(scales), scales.stride(0), _p(out), cols, rows, cols,
                                  FMT[fmt], _stream()))
    return out


def mx_gemm(a, a_scale, b, b_scale, k: int, fmt: str = "E4M3", out: str = "bf16") -> torch.Tensor:
    """C[m,n] = deq(a)[m,k] . deq(b)[n,k]^T"""
    k = index(k)
    m, n = a.size(0), b.size(0)
    return _launch("cmx_mx_gemm", a, a.stride(0), a_scale, a_scale.stride(0), b, b.stride(0), b_scale, b_scale.stride(0), (_OUT_DTYPE[out], m, n), n,
                   m, n, k, FMT[fmt], OUT[out])


def mx_to_k_major(src, src_scale, k: int, n: int):
    """codes [batch, k, n] (or [k, n]) with scales [batch, k/64, n, 2] -> K-contiguous codes [batch, n, k], scales [batch, n, k/32]."""
    _need_cuda(src, src_scale)
    assert src.is_contiguous() and src_scale.is_contiguous()
    batch = src.shape[0] if src.dim() == 3 else 1
    shape = (batch, n) if src.dim() == 3 else (n,)
    dst = torch.empty(shape + (k,), dtype=torch.uint8, device=src.device)
    dst_scale = torch.empty(shape + (k // 32,), dtype=torch.uint8, device=src.device)
    lib = _lib.load()
    _lib.check(lib.cmx_mx_to_k_major(_p(src), n, _p(src_scale), _p(dst), k, _p(dst_scale), k // 32, k, n, batch, _stream()))
    return dst, dst_scale


def mxfp4_to_k_major(src, src_scale, k: int, n: int):
    """FP4: bytes [batch, k, ceil(n/2)] (pairs along n) with scales [batch, k/64, n, 2] -> bytes [batch, n, k/2], scales [batch, n, k/32]."""
    _need_cuda(src, src_scale)
    assert src.is_contiguous() and src_scale.is_contiguous()
    batch = src.shape[0] if src.dim() == 3 else 1
    shape = (batch, n) if src.dim() == 3 else (n,)
    dst = torch.empty(shape + (k // 2,), dtype=torch.uint8, device=src.device)
    dst_scale = torch.empty(shape + (k // 32,), dtype=torch.uint8, device=src.device)
    lib = _lib.load()
    _lib.check(lib.cmx_mxfp4_to_k_major(_p(src), (n + 1) // 2, _p(src_scale), _p(dst), k // 2, _p(dst_scale), k // 32, k, n, batch,
                                        _stream()))
    return dst, dst_scale


def mx_gemm_ex(a, a_scale, b, b_scale, m: int, n: int, k: int, fmt: str = "E4M3", out: str = "bf16", trans_a: int = 0,
               trans_b: int = 1) -> torch.Tensor:
    """Dense operands in the reference's file layouts: a [m, k] (trans_a = 1: [k, m], scales [k/64, m, 2]);
    b [n, k] (trans_b = 0: [k, n], scales [k/64, n, 2])."""
    m, n, k, trans_a, trans_b = index(m), index(n), index(k), index(trans_a), index(trans_b)
    assert a.is_contiguous() and a_scale.is_contiguous() and b.is_contiguous() and b_scale.is_contiguous()
    need = _lib.load().cmx_mx_gemm_ex_workspace_bytes(m, n, k, trans_a, trans_b)
    ws = _empty(a, torch.uint8, max(need, 1))
    return _launch("cmx_mx_gemm_ex", a, a_scale, b, b_scale, (_OUT_DTYPE[out], m, n), n, m, n, k, FMT[fmt], OUT[out], trans_a, trans_b, ws)


def mx_gmm_ex(a, a_scale, b, b_scale, group_sizes, n: int, k: int, fmt: str = "E4M3", out: str = "bf16",
              trans_b: int = 1) -> torch.Tensor:
    """Grouped form: b [G, n, k] (trans_b = 0: [G, k, n], scales [G, k/64, n, 2])."""
    _need_cuda(a, a_scale, b, b_scale, group_sizes)
    assert all(t.is_contiguous() for t in (a, a_scale, b, b_scale)) and group_sizes.dtype == torch.int32
    m, g = a.shape[0], b.shape[0]
    lib = _lib.load()
    ws = torch.empty(lib.cmx_mx_gmm_ex_workspace_bytes(g, n, k, trans_b), dtype=torch.uint8, device=a.device)
    c = torch.zeros((m, n), dtype=_OUT_DTYPE[out], device=a.device)
    _lib.check(lib.cmx_mx_gmm_ex(_p(a), _p(a_scale), _p(b), _p(b_scale), _p(c), n, _p(group_sizes), g, m, n, k, FMT[fmt],
                                 OUT[out], trans_b, _p(ws), _stream()))
    return c


def int8_quant_scatter(x: torch.Tensor, src2sorted, top_k: int = 1):
    """x bf16 [tokens, k] -> (codes int8 [tokens*top_k, k], scales fp32 [tokens*top_k]); row t goes to src2sorted[t*top_k + r]."""
    top_k = index(top_k)
    assert x.dim() == 2 and x.element_size() == 2
    tokens, k = x.shape
    pitch, step = x.stride()
    assert step == 1
    _no_new(src2sorted)
    return _launch("cmx_int8_quant_scatter", x, pitch, src2sorted, (torch.int8, tokens * top_k, k), k, (torch.float32, tokens * top_k), tokens, k, top_k)


def int8_gmm_dequant_swiglu(a, token_scale, b, channel_scale, group_sizes, n: int, k: int, trans_b: int = 0,
                            out: str = "fp32", scale_stride: int = 1, c=None) -> torch.Tensor:
    """a int8 [rows, k]; b int8 [G, k, n] (trans_b = 0) or [G, n, k] (trans_b = 1); channel_scale fp32 [G*n*scale_stride]."""
    n, k, trans_b, scale_stride = index(n), index(k), index(trans_b), index(scale_stride)
    assert a.is_contiguous() and b.is_contiguous() and group_sizes.dtype == torch.int32
    _no_new(token_scale, channel_scale)
    rows, g = a.size(0), b.size(0)
    ws = _empty(a, torch.uint8, _lib.load().cmx_int8_gmm_workspace_bytes(g, n, k, trans_b))
    if c is None:
        c = torch.zeros((rows, n // 2), dtype=_OUT_DTYPE[out], device=a.device)
    _launch("cmx_int8_gmm_dequant_swiglu", a, k, token_scale, b, channel_scale, scale_stride, _brought(c), c.stride(0), OUT[out], group_sizes, g, rows, n, k,
            trans_b, ws)
    return c


def gmm_workspace(groups: int, device) -> torch.Tensor:
    lib = _lib.load()
    return torch.empty(lib.cmx_mx_gmm_workspace_bytes(groups), dtype=torch.uint8, device=device)


class PretiledWeights:
    """Expert weights [groups, n, k] (8-bit codes) in the tiled order of cmx_mx_pretile_weights; ``pair_gate_up``
    says which of the two grouped matmuls the tiling is for (True: mx_gmm_swiglu_quant, False: mx_gmm)."""

    def __init__(self, data: torch.Tensor, groups: int, n: int, k: int, pair_gate_up: bool):
        self.data, self.groups, self.n, self.k, self.pair_gate_up = data, groups, n, k, pair_gate_up

    @property
    def shape(self):
        return (self.groups, self.n, self.k)


def pretile_weights(b: torch.Tensor, pair_gate_up: bool) -> PretiledWeights:
    """b u8 [G, n, k] dense -> PretiledWeights (one pass over the weights; meant for weight-load time)."""
    _need_cuda(b)
    assert b.dtype == torch.uint8 and b.dim() == 3 and b.is_contiguous()
    g, n, k = b.shape
    lib = _lib.load()
    nbytes = lib.cmx_mx_pretiled_weight_bytes(g, n, k, int(pair_gate_up))
    if nbytes == 0:
        raise ValueError("pre-tiled weights need k % 512 == 0 (and n % 64 == 0 for gate|up weights)")
    out = torch.empty(nbytes, dtype=torch.uint8, device=b.device)
    _lib.check(lib.cmx_mx_pretile_weights(_p(b), _p(out), g, n, k, int(pair_gate_up), _stream()))
    return PretiledWeights(out, g, n, k, bool(pair_gate_up))


def _weights(b, pair_gate_up: bool):
    """(tensor, pretiled?) of a weight argument: a dense tensor or PretiledWeights of the matching kind."""
    if isinstance(b, PretiledWeights):
        assert b.pair_gate_up == pair_gate_up, "weights were pre-tiled for the other grouped matmul"
        return b.data, True
    assert b.is_contiguous()
    return b, False


def mx_gmm(a, a_scale, b, b_scale, group_sizes, k: int, fmt: str = "E4M3", out: str = "bf16", c=None, workspace=None):
    """a [m_total, k], b [G, n, k] (dense tensor or PretiledWeights), group_sizes int32 [G] on device -> c [m_total, n]
    (rows past the groups untouched)."""
    k = index(k)
    assert b_scale.is_contiguous() and group_sizes.dtype == torch.int32
    bd, tiled = _weights(b, False)
    m, (g, n) = a.size(0), b.shape[:2]
    if c is None:
        c = torch.zeros((m, n), dtype=_OUT_DTYPE[out], device=a.device)
    if workspace is None:
        workspace = gmm_workspace(g, a.device)
    _launch("cmx_mx_gmm_pretiled" if tiled else "cmx_mx_gmm", a, a.stride(0), a_scale, a_scale.stride(0), _brought(bd), b_scale, _brought(c),
            c.stride(0), group_sizes, g, m, n, k, FMT[fmt], OUT[out], _brought(workspace))
    return c


def mx_gmm_swiglu_quant(a, a_scale, b, b_scale, group_sizes, k: int, want_bf16: bool = False, workspace=None,
                        outs=None):
    """GMM1 + SwiGLU + MX requant.  b [G, n, k] (gate rows then up rows; dense tensor or PretiledWeights).
    Returns (codes [m, n/2], scales, act_bf16|None)."""
    k = index(k)
    assert b_scale.is_contiguous() and group_sizes.dtype == torch.int32
    bd, tiled = _weights(b, True)
    m, (g, n) = a.size(0), b.shape[:2]
    half = n // 2
    if outs is None:
        codes = torch.zeros((m, half), dtype=torch.uint8, device=a.device)
        scales = torch.zeros((m, scale_cols(half)), dtype=torch.uint8, device=a.device)
    else:
        codes, scales = outs
    act = torch.zeros((m, half), dtype=torch.bfloat16, device=a.device) if want_bf16 else None
    if workspace is None:
        workspace = gmm_workspace(g, a.device)
    _launch("cmx_mx_gmm_swiglu_quant_pretiled" if tiled else "cmx_mx_gmm_swiglu_quant", a, a.stride(0), a_scale, a_scale.stride(0), _brought(bd),
            b_scale, _brought(codes), codes.stride(0), _brought(scales), scales.stride(0), act, group_sizes, g, m, n, k, _brought(workspace))
    return codes, scales, act


def mx_gmm_swiglu_quant_noalloc(a, a_scale, b, b_scale, group_sizes, k: int, codes, scales, act=None) -> None:
    """cmx_mx_gmm_swiglu_quant_noalloc: the caller brings every buffer (codes [m, n/2], scales, optional bf16 act);
    neither this wrapper nor the library allocates anything."""
    _need_cuda(a, a_scale, b, b_scale, group_sizes, codes, scales)
    assert b.is_contiguous() and b_scale.is_contiguous() and group_sizes.dtype == torch.int32
    m, (g, n) = a.shape[0], b.shape[:2]
    lib = _lib.load()
    _lib.check(lib.cmx_mx_gmm_swiglu_quant_noalloc(_p(a), a.stride(0), _p(a_scale), a_scale.stride(0), _p(b), _p(b_scale),
                                                   _p(codes), codes.stride(0), _p(scales), scales.stride(0), _p(act),
                                                   _p(group_sizes), g, m, n, k, _stream()))


def init() -> None:
    """cmx_init on the current device."""
    _lib.check(_lib.load().cmx_init())


def moe_init_routing(expert_idx: torch.Tensor, experts: int):
    """expert_idx int32 [T, topK] -> (sorted2src, src2sorted, counts) int32."""
    experts = index(experts)
    assert expert_idx.dtype == torch.int32 and expert_idx.is_contiguous()
    t, top_k = expert_idx.shape
    routes = t * top_k
    ws = _empty(expert_idx, torch.uint8, _lib.load().cmx_moe_routing_workspace_bytes(routes, experts))
    return _launch("cmx_moe_init_routing", expert_idx, t, top_k, experts, (torch.int32, routes), (torch.int32, routes), (torch.int32, experts), ws)


def quant_scatter(x: torch.Tensor, src2sorted: torch.Tensor, top_k: int, packed: bool = False, out=None):
    """x bf16 [T, k] -> rows quantised once and written to their top_k destinations.
    packed=False: (codes [T*topK, k], scales [T*topK, RoundUp2(k/32)]), zeros in rows that no route is sent to;
    packed=True: one buffer [T*topK, packed_row_bytes(k)] = codes | scales | pad (``out``: a caller's zeroed buffer
    of that shape)."""
    top_k = index(top_k)
    _need_cuda(x, src2sorted)
    t, k = x.shape
    rows = t * top_k
    lib = _lib.load()
    if packed:
        rb = lib.cmx_packed_row_bytes(k)
        buf = torch.zeros((rows, rb), dtype=torch.uint8, device=x.device) if out is None else out
        assert buf.shape == (rows, rb) and buf.dtype == torch.uint8 and buf.is_contiguous()
        _lib.check(lib.cmx_quant_scatter(_p(x), x.stride(0), _p(src2sorted), _p(buf), rb, buf.data_ptr() + k, rb, t, k,
                                         top_k, _stream()))
        return buf
    scols = scale_cols(k)
    return _launch("cmx_quant_scatter_zeroed", x, x.stride(0), src2sorted, (torch.uint8, rows, k), k, (torch.uint8, rows, scols), scols, t, k, top_k)


def moe_token_unpermute(y: torch.Tensor, src2sorted: torch.Tensor, probs: torch.Tensor) -> torch.Tensor:
    """y bf16 [rows, h]; probs fp32 [T, topK] -> bf16 [T, h]."""
    _need_cuda(y, src2sorted, probs)
    assert probs.dtype == torch.float32 and probs.is_contiguous()
    t, top_k = probs.shape
    rows, h = y.shape
    out = torch.empty((t, h), dtype=y.dtype, device=y.device)
    lib = _lib.load()
    _lib.check(lib.cmx_moe_token_unpermute(_p(y), y.stride(0), rows, _p(src2sorted), _p(probs), _p(out), h, t, h, top_k,
                                           _stream()))
    return out


def ffn_workspace_bytes(m: int, k: int, n: int, experts: int, top_k: int) -> int:
    return _lib.load().catccos_ascend950_dispatch_ffn_combine_workspace_bytes(m, k, n, experts, top_k, 1)


def ffn_workspace_layout(m: int, k: int, n: int, experts: int, top_k: int) -> dict:
    lay = _lib.FfnWorkspaceLayout()
    _lib.check(_lib.load().cmx_ffn_workspace_layout_get(m, k, n, experts, top_k, lay))
    return {f: getattr(lay, f) for f, _ in lay._fields_}


def dispatch_ffn_combine(x, expert_idx, gate_weight, w1, w1_scale, w2, w2_scale, workspace=None, out=None):
    """torch.ops.catccos.ascend950_dispatch_ffn_combine(x, expert_idx, gate_weight, w1, w1_scale, w2, w2_scale)
    on one GPU: x bf16 [m,k]; expert_idx int32 [m,topK]; gate_weight fp32 [m,topK];
    w1 [E,n,k] + w1_scale [E,n,k/32]; w2 [E,k,n/2] + w2_scale [E,k,n/64] -> bf16 [m,k].
    w1 and w2 may both be PretiledWeights (w1 tiled with pair_gate_up=True, w2 with False): same result, through
    cmx_dispatch_ffn_combine_pretiled."""
    _need_cuda(x, expert_idx, gate_weight, w1_scale, w2_scale)
    m, k = x.shape
    e, n = w1.shape[:2]
    top_k = expert_idx.shape[1]
    for t in (x, expert_idx, gate_weight, w1_scale, w2_scale):
        assert t.is_contiguous()
    w1d, tiled1 = _weights(w1, True)
    w2d, tiled2 = _weights(w2, False)
    assert tiled1 == tiled2, "pre-tile both weight tensors or neither"
    if workspace is None:
        workspace = _empty(x, torch.uint8, ffn_workspace_bytes(m, k, n, e, top_k))
    if out is None:
        out = _empty(x, x.dtype, m, k)
    w1d, w2d, out_at, workspace = _brought(w1d), _brought(w2d), _brought(out), _brought(workspace)
    entries = _lib.entries()
    if tiled1:
        rc = _run(entries["cmx_dispatch_ffn_combine_pretiled"], _stream(), x, expert_idx, gate_weight, w1d, w1_scale, w2d, w2_scale, out_at, workspace,
                  m, k, n, e, top_k)
    else:
        rc = _run(entries["catccos_ascend950_dispatch_ffn_combine"], 0, _stream(), 0, x, expert_idx, gate_weight, w1d, w1_scale, w2d, w2_scale, out_at,
                  workspace, None, m, k, n, e, top_k, 1)
    _lib.check(rc)
    return out
