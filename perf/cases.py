"""The calls that the performance of this library is measured on.

Seven paths, each through the Python entry points of ``catccos_amd`` (thin wrappers of the C ABI) in the order in which a
program calls them:

  quant     bf16 activations -> MX codes and scales (``ops.mx_quant``)
  linear    bf16 activations -> MX -> dense matmul with resident MX weights -> 16-bit output (``mx_quant``, ``mx_gemm``)
  kslow     the same with the weights stored [K, N], K the slow axis, as the reference's generators write them with
            trans_b = 0 (``mx_quant``, ``mx_gemm_ex``)
  gmm1      MoE up-projection of one device: expert sort, quantise + scatter, grouped matmul with fused SwiGLU and MX requant
            (``moe_init_routing``, ``quant_scatter``, ``mx_gmm_swiglu_quant``)
  int8      the same operator in the reference's INT8 arithmetic (``moe_init_routing``, ``int8_quant_scatter``,
            ``int8_gmm_dequant_swiglu``; weights K-contiguous, as the host operator keeps them)
  fp4       MXFP4 W4A4 grouped matmul on expert-sorted rows (``mx_quant`` to E2M1, ``mx_gmm``)
  ffn       the whole MoE FFN of one device (``ops.dispatch_ffn_combine`` on weights tiled once at load time, or the torch
            operator ``catccos.ascend950_dispatch_ffn_combine`` on row-major weights)

Weights, workspaces and large output buffers are made once, as a serving or training program keeps them; everything that
depends on the activations happens in ``run``.
"""
from __future__ import annotations

import math

import torch

from catccos_amd import ops

DEV = "cuda"


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # activations of one layer on their way into a matmul: the quantizer alone, 4096 tokens x 7168
        {"name": "quant 4096x7168", "path": "quant", "rows": 4096, "cols": 7168, "fmt": "E4M3"},
        # one projection at decode: a handful of tokens against 29 MB of weights
        {"name": "linear decode", "path": "linear", "m": 16, "n": 4096, "k": 7168, "fmt": "E4M3", "out": "bf16"},
        # a small odd-sized projection (the reference's own dense test shape 1000 x 960 x 1000, E5M2)
        {"name": "linear odd", "path": "linear", "m": 1000, "n": 1000, "k": 960, "fmt": "E5M2", "out": "bf16"},
        # the dense matmul at prefill size
        {"name": "linear prefill", "path": "linear", "m": 8192, "n": 4096, "k": 7168, "fmt": "E4M3", "out": "bf16"},
        # a mid-sized batch on weights stored [K, N] (the reference's trans_b = 0 setting)
        {"name": "linear k-slow weights", "path": "kslow", "m": 1024, "n": 4096, "k": 7168, "fmt": "E4M3", "out": "bf16"},
        # dispatch_gmm_dequant_swiglu's local work: 4096 tokens, top-8 of 16 experts with Zipf load, two experts empty
        {"name": "moe gmm1 prefill", "path": "gmm1", "tokens": 4096, "experts": 16, "top_k": 8, "k": 7168, "n": 4096},
        # the same operator in INT8
        {"name": "moe int8 prefill", "path": "int8", "tokens": 4096, "experts": 16, "top_k": 8, "k": 7168, "n": 4096},
        # FP4 grouped matmul: a large batch, and one decode step of 64 tokens
        {"name": "moe fp4 prefill", "path": "fp4", "tokens": 8192, "experts": 32, "top_k": 8, "k": 7168, "n": 4096},
        {"name": "moe fp4 decode", "path": "fp4", "tokens": 64, "experts": 32, "top_k": 8, "k": 7168, "n": 4096},
        # the whole FFN, 256 experts: prefill and one decode step, on weights tiled at load time
        {"name": "ffn prefill", "path": "ffn", "tokens": 8192, "experts": 256, "top_k": 8, "k": 7168, "n": 4096, "tiled": True},
        {"name": "ffn decode", "path": "ffn", "tokens": 32, "experts": 256, "top_k": 8, "k": 7168, "n": 4096, "tiled": True},
        # the torch operator on row-major weights, an odd number of tokens
        {"name": "ffn torch op", "path": "ffn", "tokens": 777, "experts": 32, "top_k": 8, "k": 7168, "n": 4096, "tiled": False},
    ]


def _log_int(rng, lo, hi):
    """A whole number from [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _step(rng, lo, hi, by):
    """A multiple of `by` from [lo, hi], its logarithm uniform."""
    return min(hi // by * by, max(-(-lo // by) * by, round(_log_int(rng, lo, hi) / by) * by))


def draw(rng):
    path = rng.choice(("quant", "linear", "linear", "kslow", "gmm1", "int8", "fp4", "ffn", "ffn"))
    if path == "quant":
        # rows of any number, hidden sizes in whole MX blocks
        return {"path": path, "rows": _log_int(rng, 16, 16384), "cols": _step(rng, 512, 8192, 32),
                "fmt": rng.choice(("E4M3", "E4M3", "E5M2", "E2M1"))}
    if path in ("linear", "kslow"):
        # from one token to a prefill batch; K-slow weights come in whole pairs of K blocks
        by = 32 if path == "linear" else 64
        return {"path": path, "m": _log_int(rng, 1, 8192 if path == "linear" else 4096), "n": _step(rng, 512, 8192, 8),
                "k": _step(rng, 512, 8192, rng.choice((by, 128, 512))), "fmt": rng.choice(("E4M3", "E4M3", "E5M2")),
                "out": rng.choice(("bf16", "bf16", "fp16"))}
    if path == "gmm1":
        return {"path": path, "tokens": _log_int(rng, 8, 4096), "experts": rng.choice((8, 16, 32)), "top_k": rng.choice((2, 4, 6, 8)),
                "k": _step(rng, 1024, 7168, rng.choice((128, 512))), "n": _step(rng, 1024, 4096, 256)}
    if path == "int8":
        return {"path": path, "tokens": _log_int(rng, 8, 4096), "experts": rng.choice((8, 16, 32)), "top_k": rng.choice((2, 4, 6, 8)),
                "k": _step(rng, 1024, 7168, 128), "n": _step(rng, 1024, 4096, 64)}
    if path == "fp4":
        return {"path": path, "tokens": _log_int(rng, 8, 8192), "experts": rng.choice((8, 16, 32)), "top_k": rng.choice((2, 4, 6, 8)),
                "k": _step(rng, 1024, 7168, rng.choice((256, 512))), "n": _step(rng, 1024, 7168, 64)}
    tiled = rng.random() < 0.6
    experts = rng.choice((16, 32, 64, 128, 256) if tiled else (8, 16, 32, 64))
    return {"path": path, "tokens": _log_int(rng, 1, 4096), "experts": experts, "top_k": rng.choice((2, 4, 6, 8)),
            "k": _step(rng, 1024, 7168, 512 if tiled else 256), "n": _step(rng, 1024, 4096, 1024 if tiled else 512), "tiled": tiled}


# ------------------------------------------------------------------------------------------------ their inputs
def _activations(gen, rows, cols):
    """bf16 N(0, 1) with 0.1 % outliers a hundred times as large, as activations have them."""
    x = torch.randn((rows, cols), generator=gen, device=DEV)
    x.mul_(1.0 + 99.0 * (torch.rand((rows, cols), generator=gen, device=DEV) < 1e-3))
    return x.to(torch.bfloat16)


def _weights(gen, experts, n, k, std, fmt):
    """[experts, n, k] MX weights: N(0, std) rounded by table, as weights are quantised off line."""
    shape = (experts, n, k // 2 if fmt == "E2M1" else k)
    codes = torch.empty(shape, dtype=torch.uint8, device=DEV)
    scales = torch.empty((experts, n, ops.scale_cols(k)), dtype=torch.uint8, device=DEV)
    for e in range(experts):
        codes[e], scales[e] = ops.mx_quant(torch.randn((n, k), generator=gen, device=DEV).mul_(std).to(torch.bfloat16), fmt, "lut")
    return codes, scales


def _zipf_experts(gen, tokens, experts, top_k):
    """int32 [tokens, top_k]: distinct experts per token with probabilities 1 / rank^1.1, the two last-ranked experts never
    chosen when there are enough others."""
    p = 1.0 / torch.arange(1, experts + 1, device=DEV, dtype=torch.float32) ** 1.1
    if experts - 2 >= top_k:
        p[experts - 2:] = 0.0
    p = p[torch.randperm(experts, generator=gen, device=DEV)]
    gumbel = -torch.log(-torch.log(torch.rand((tokens, experts), generator=gen, device=DEV).clamp_(1e-20, 1.0 - 1e-7)))
    return (torch.log(p) + gumbel).topk(top_k, dim=1).indices.to(torch.int32).contiguous()


def _softmax_experts(gen, tokens, experts, top_k):
    """(int32 experts, fp32 weights) [tokens, top_k]: top-k of a softmax over N(0, 1) logits, renormalised."""
    p, idx = torch.softmax(torch.randn((tokens, experts), generator=gen, device=DEV), dim=1).topk(top_k, dim=1)
    return idx.to(torch.int32).contiguous(), (p / p.sum(dim=1, keepdim=True)).contiguous()


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    c, s = case, {"case": case}
    if c["path"] == "quant":
        s["x"] = _activations(gen, c["rows"], c["cols"])
    elif c["path"] in ("linear", "kslow"):
        s["x"] = _activations(gen, c["m"], c["k"])
        w, ws = _weights(gen, 1, c["n"], c["k"], 0.02, c["fmt"])
        s["w"], s["ws"] = w[0], ws[0]
        if c["path"] == "kslow":
            s["w"] = w[0].t().contiguous()                                              # [k, n]
            s["ws"] = ws[0].view(c["n"], c["k"] // 64, 2).permute(1, 0, 2).contiguous()  # [k / 64, n, 2]
    elif c["path"] in ("gmm1", "int8"):
        rows = c["tokens"] * c["top_k"]
        s["x"] = _activations(gen, c["tokens"], c["k"])
        s["idx"] = _zipf_experts(gen, c["tokens"], c["experts"], c["top_k"])
        if c["path"] == "gmm1":
            s["w"], s["ws"] = _weights(gen, c["experts"], c["n"], c["k"], 0.02, "E4M3")
            s["work"] = ops.gmm_workspace(c["experts"], DEV)
            s["outs"] = (torch.empty((rows, c["n"] // 2), dtype=torch.uint8, device=DEV),
                         torch.zeros((rows, ops.scale_cols(c["n"] // 2)), dtype=torch.uint8, device=DEV))
        else:
            s["w"] = torch.randint(-127, 128, (c["experts"], c["n"], c["k"]), dtype=torch.int8, device=DEV, generator=gen)
            s["channel"] = torch.rand((c["experts"] * c["n"],), device=DEV, generator=gen) * (2.0 * 0.06 / 127)
            s["out"] = torch.empty((rows, c["n"] // 2), dtype=torch.float32, device=DEV)
    elif c["path"] == "fp4":
        rows = c["tokens"] * c["top_k"]
        s["x"] = _activations(gen, rows, c["k"])
        idx = _zipf_experts(gen, c["tokens"], c["experts"], c["top_k"])
        s["counts"] = torch.bincount(idx.view(-1).long(), minlength=c["experts"]).to(torch.int32)
        s["w"], s["ws"] = _weights(gen, c["experts"], c["n"], c["k"], 0.02, "E2M1")
        s["work"] = ops.gmm_workspace(c["experts"], DEV)
        s["out"] = torch.empty((rows, c["n"]), dtype=torch.bfloat16, device=DEV)
    else:
        s["x"] = torch.randn((c["tokens"], c["k"]), generator=gen, device=DEV).to(torch.bfloat16)
        s["idx"], s["gate"] = _softmax_experts(gen, c["tokens"], c["experts"], c["top_k"])
        w1, s["w1s"] = _weights(gen, c["experts"], c["n"], c["k"], 0.02, "E4M3")
        if c["tiled"]:
            s["w1"] = ops.pretile_weights(w1, True)
            del w1
            w2, s["w2s"] = _weights(gen, c["experts"], c["k"], c["n"] // 2, 0.02, "E4M3")
            s["w2"] = ops.pretile_weights(w2, False)
            s["work"] = torch.empty(ops.ffn_workspace_bytes(c["tokens"], c["k"], c["n"], c["experts"], c["top_k"]), dtype=torch.uint8,
                                    device=DEV)
            s["out"] = torch.empty_like(s["x"])
        else:
            import catccos_amd.torch_op  # noqa: F401  (registers torch.ops.catccos)
            torch.ops.catccos.init(0, 1, 1 << 30, "tcp://127.0.0.1:1")
            w2, w2s = _weights(gen, c["experts"], c["k"], c["n"] // 2, 0.02, "E4M3")
            s["w1"], s["w2"] = w1.view(torch.float8_e4m3fn), w2.view(torch.float8_e4m3fn)
            s["w1s"], s["w2s"] = s["w1s"].view(torch.float8_e8m0fnu), w2s.view(torch.float8_e8m0fnu)
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    c = s["case"]
    if c["path"] == "quant":
        return ops.mx_quant(s["x"], c["fmt"])
    if c["path"] == "linear":
        a, a_s = ops.mx_quant(s["x"], c["fmt"])
        return ops.mx_gemm(a, a_s, s["w"], s["ws"], c["k"], c["fmt"], c["out"])
    if c["path"] == "kslow":
        a, a_s = ops.mx_quant(s["x"], c["fmt"])
        return ops.mx_gemm_ex(a, a_s, s["w"], s["ws"], c["m"], c["n"], c["k"], c["fmt"], c["out"], trans_a=0, trans_b=0)
    if c["path"] == "gmm1":
        _, dest, counts = ops.moe_init_routing(s["idx"], c["experts"])
        a, a_s = ops.quant_scatter(s["x"], dest, c["top_k"])
        codes, scales, _ = ops.mx_gmm_swiglu_quant(a, a_s, s["w"], s["ws"], counts, c["k"], workspace=s["work"], outs=s["outs"])
        return codes, scales
    if c["path"] == "int8":
        _, dest, counts = ops.moe_init_routing(s["idx"], c["experts"])
        a, token_scale = ops.int8_quant_scatter(s["x"], dest, c["top_k"])
        return ops.int8_gmm_dequant_swiglu(a, token_scale, s["w"], s["channel"], counts, c["n"], c["k"], 1, "fp32", c=s["out"])
    if c["path"] == "fp4":
        a, a_s = ops.mx_quant(s["x"], "E2M1")
        return ops.mx_gmm(a, a_s, s["w"], s["ws"], s["counts"], c["k"], "E2M1", "bf16", c=s["out"], workspace=s["work"])
    if c["tiled"]:
        return ops.dispatch_ffn_combine(s["x"], s["idx"], s["gate"], s["w1"], s["w1s"], s["w2"], s["w2s"], workspace=s["work"], out=s["out"])
    return torch.ops.catccos.ascend950_dispatch_ffn_combine(s["x"], s["idx"], s["gate"], s["w1"], s["w1s"], s["w2"], s["w2s"])


# ------------------------------------------------------------------------------------------------ what it cannot do without
def _active(tokens, experts, top_k):
    """Experts that get a row, on average, when every token takes top_k of them at random (a Zipf load uses somewhat fewer when
    there are few tokens)."""
    return experts * (1.0 - (1.0 - top_k / experts) ** tokens)


def work(case):
    c, mx = case, 1.0 + 1.0 / 32
    if c["path"] == "quant":
        bits = 0.5 if c["fmt"] == "E2M1" else 1.0
        return {"bytes": c["rows"] * c["cols"] * (2 + bits + 1 / 32), "flops": 0}
    if c["path"] in ("linear", "kslow"):
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 2 * m * k + n * k * mx + 2 * m * n, "flops": 2 * m * n * k}
    rows, k, n, e = c["tokens"] * c["top_k"], c["k"], c["n"], c["experts"]
    if c["path"] == "ffn":
        used = _active(c["tokens"], e, c["top_k"])
        return {"bytes": 2 * 2 * c["tokens"] * k + used * 1.5 * n * k * mx + 8 * rows, "flops": 3 * rows * n * k}
    used = min(_active(c["tokens"], e, c["top_k"]), e - 2 if e - 2 >= c["top_k"] else e)
    if c["path"] == "gmm1":
        return {"bytes": 2 * c["tokens"] * k + used * n * k * mx + rows * (n // 2) * mx + 4 * rows, "flops": 2 * rows * n * k}
    if c["path"] == "int8":
        return {"bytes": 2 * c["tokens"] * k + used * n * (k + 4) + 4 * rows * (n // 2) + 4 * rows, "flops": 2 * rows * n * k}
    return {"bytes": 2 * rows * k + used * n * k * (0.5 + 1 / 32) + 2 * rows * n, "flops": 2 * rows * n * k}


def tolerance(case):
    """About four times what each path differs from itself computed in 64 bits from the same codes and rounded where the path
    rounds (2-norm and largest difference, share of codes)."""
    path = case["path"]
    if path == "quant":
        return "exact"                                     # codes and scale bytes
    if path in ("linear", "kslow"):
        # seen: bf16 5.7e-4 (one rounding in ten goes to the other neighbour: the matrix cores align the products of an
        # instruction before they add them), one unit in the last place at most; fp16 1.5e-4
        return {"rel": 2.3e-3, "max": 3e-2} if case["out"] == "bf16" else {"rel": 6e-4, "max": 4e-3}
    if path == "gmm1":
        return {"rel": 0.0, "differ": 1e-2}                # seen: 5e-3 of the codes, 1e-4 of the scales
    if path == "int8":
        return {"rel": 3e-5, "max": 4e-3}                  # whole-number sums; seen: 8e-6, the fp16 step of one value in max
    if path == "fp4":
        return {"rel": 2e-4, "max": 3e-2}                  # 32-bit sums of short products: one output in ten thousand rounds the other way
    return {"rel": 9e-3, "max": 0.15}                      # seen: 2.3e-3 and 0.04, codes of the inner activations among the causes
