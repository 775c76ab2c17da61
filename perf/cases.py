"""Workloads of the MXFP / minifloat path: layers and functional linears from one decode row to a long prefill, a SwiGLU
block, attention products, and the casts themselves, in the data types and formats they are used with.

A case is a dict of plain values; ``kind`` says which entry point it goes through:

  linear        an ``MXFPLinearPTQ`` / ``MinifloatLinearPTQ`` layer's forward (the layer keeps its quantised weight)
  linear_call   the functional ``mxfp_linear`` on weight components (nothing kept between calls)
  mlp           a SwiGLU block of two layers: stacked gate / up, then ``forward_swiglu`` of the down layer
  matmul        ``mxfp_matmul`` over batch x heads: queries against keys, or probabilities against values
  mxfp_cast     extract + compose, or the fused quantise-dequantise, blocks along the last axis or down the rows
  minifloat_cast  the same for element-wise minifloat formats
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("mase-triton_amd"))

import mase_hip.minifloat.functional as MF  # noqa: E402
import mase_hip.minifloat.meta as mf_meta  # noqa: E402
import mase_hip.mxfp.functional as MX  # noqa: E402
import mase_hip.mxfp.meta as mx_meta  # noqa: E402
from mase_hip.minifloat.layers import MinifloatLinearPTQ  # noqa: E402
from mase_hip.mxfp.layers import MXFPLinearPTQ  # noqa: E402

DEV = "cuda:0"
MXFP = {"E4M3": mx_meta.MXFP8_E4M3_fn, "E5M2": mx_meta.MXFP8_E5M2_fn, "E2M3": mx_meta.OCP_MXFP6_E2M3,
        "E3M2": mx_meta.OCP_MXFP6_E3M2, "E2M1": mx_meta.OCP_MXFP4_E2M1}
MINIFLOAT = {"E4M3": mf_meta.FP8_E4M3_fn, "E5M2": mf_meta.FP8_E5M2_fn, "E2M3": mf_meta.FP6_E2M3_fn,
             "E3M2": mf_meta.FP6_E3M2_fn, "E2M1": mf_meta.FP4_E2M1_fn}
SIZE = {"bfloat16": 2, "float16": 2, "float32": 4}


def listed():
    return [
        # one token of one sequence through a square projection of a 4096-wide decoder: the smallest call there is
        dict(name="decode_1_row", kind="linear", family="mxfp", layer="XqWqB", rows=1, k=4096, n=4096, x_fmt="E4M3", w_fmt="E4M3",
             dtype="bfloat16", bias=False),
        # 48 sequences decoding together, the down projection of a Llama-3-8B MLP with 4-bit weights (long K, few columns)
        dict(name="decode_48_rows_down", kind="linear", family="mxfp", layer="XqWqB", rows=48, k=14336, n=4096, x_fmt="E4M3", w_fmt="E2M1",
             dtype="bfloat16", bias=False),
        # a serving step of 200 tokens (a large decode batch, or a short chunk of a prompt) through an up projection
        dict(name="batch_200_rows", kind="linear", family="mxfp", layer="XqWqB", rows=200, k=4096, n=14336, x_fmt="E4M3", w_fmt="E3M2",
             dtype="bfloat16", bias=True),
        # weight-only quantisation: dense bf16 activations of a few sequences against 4-bit weights
        dict(name="weight_only_12_rows", kind="linear", family="mxfp", layer="XWqB", rows=12, k=4096, n=14336, x_fmt="E4M3", w_fmt="E2M1",
             dtype="bfloat16", bias=False),
        # the benchmark's product: a long prefill through the functional call, weight given as components
        dict(name="linear_call_16384", kind="linear_call", rows=16384, k=4096, n=14336, x_fmt="E4M3", w_fmt="E4M3"),
        # a whole Llama-3-8B SwiGLU block over 4 x 2048 tokens, 6-bit weights and 8-bit activations: the largest
        dict(name="mlp_8192", kind="mlp", rows=8192, hidden=4096, inter=14336, x_fmt="E4M3", w_fmt="E3M2"),
        # attention scores of 2 sequences x 32 heads, both operands quantised; the keys come as a transposed view, as in a model
        dict(name="attention_qk_1000", kind="matmul", product="qk", batch=2, heads=32, q_len=1000, kv_len=1000, head_dim=128, fmt="E4M3"),
        # an activation matrix to components and back (MXFP8), the 4096 x 4096 round trip of the benchmark
        dict(name="mxfp8_round_trip_bf16", kind="mxfp_cast", op="round_trip", rows=4096, cols=4096, block_dim=-1, fmt="E4M3", dtype="bfloat16"),
        # an fp32 master weight rounded to MXFP4 (an MLP weight; zero blocks and a few inf / NaN among them)
        dict(name="mxfp4_qdq_f32", kind="mxfp_cast", op="qdq", rows=14336, cols=4096, block_dim=-1, fmt="E2M1", dtype="float32"),
        # fp16 matrix whose blocks run down the rows (the right operand of a product)
        dict(name="mxfp8_rows_f16", kind="mxfp_cast", op="round_trip", rows=2976, cols=4096, block_dim=0, fmt="E4M3", dtype="float16"),
        # element-wise FP8 rounding of 2^24 fp32 values with outliers, zeros and subnormals
        dict(name="fp8_qdq_f32", kind="minifloat_cast", op="qdq", count=1 << 24, fmt="E4M3", dtype="float32"),
        # codes of a bf16 tensor with an odd number of elements, and back
        dict(name="fp8_round_trip_bf16_odd", kind="minifloat_cast", op="round_trip", count=3_000_001, fmt="E5M2", dtype="bfloat16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, ragged=True):
    """(in, out) features: the listed layers' and generic ones, most of them multiples of 128, some only of 32 (in) or odd (out)."""
    if rng.random() < 0.4:
        return rng.choice([(4096, 4096), (4096, 14336), (14336, 4096), (4096, 1024), (4096, 12288), (2048, 8192), (8192, 2048)])
    if not ragged or rng.random() < 0.7:
        k = 128 * _log(rng, 6, 112)
        return k, 128 * _log(rng, 6, min(112, 4096 * 14336 // (128 * k)))
    return 32 * _log(rng, 24, 256), _log(rng, 500, 8192)


_FMTS = ["E4M3", "E4M3", "E3M2", "E2M3", "E2M1", "E5M2"]


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["linear_call", "linear_call", "mlp", "matmul", "matmul", "mxfp_cast", "mxfp_cast", "mxfp_cast",
                                        "minifloat_cast", "minifloat_cast"])
    if kind == "linear":
        k, n = _features(rng)
        rows = _log(rng, 1, 4096)
        dtype = rng.choice(["bfloat16"] * 7 + ["float32", "float32", "float16"])
        layer = rng.choice(["XqWqB", "XqWqB", "XWqB"]) if dtype == "bfloat16" else "XqWqB"
        return dict(kind=kind, family=rng.choice(["mxfp", "mxfp", "minifloat"]), layer=layer, rows=rows, k=k, n=n, x_fmt=rng.choice(_FMTS),
                    w_fmt=rng.choice(_FMTS), dtype=dtype, bias=rng.random() < 0.4)
    if kind == "linear_call":
        k, n = _features(rng, ragged=False)
        rows = _log(rng, 16, 16384)
        return dict(kind=kind, rows=rows, k=k, n=n, x_fmt="E4M3", w_fmt=rng.choice(_FMTS[:-1] if rows > 8192 else _FMTS))
    if kind == "mlp":
        hidden, inter = rng.choice([(4096, 14336), (2048, 8192), (1024, 4096), (4096, 12288)])
        return dict(kind=kind, rows=_log(rng, 1, 8192), hidden=hidden, inter=inter, x_fmt="E4M3", w_fmt=rng.choice(["E4M3", "E3M2", "E2M3", "E2M1"]))
    if kind == "matmul":
        product = rng.choice(["qk", "pv"])
        kv_len = _log(rng, 64, 2048) if product == "qk" else 32 * _log(rng, 2, 64)
        q_len = kv_len if rng.random() < 0.7 else _log(rng, 1, 64)
        return dict(kind=kind, product=product, batch=rng.choice([1, 1, 2, 4]), heads=rng.choice([8, 16, 32]), q_len=q_len, kv_len=kv_len,
                    head_dim=rng.choice([64, 128]), fmt=rng.choice(_FMTS))
    dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float32", "float32"])
    op = rng.choice(["round_trip", "qdq"])
    if kind == "mxfp_cast":
        block_dim = rng.choice([-1, -1, 0])
        total = _log(rng, 1 << 12, 5 << 23)
        cols = 32 * _log(rng, 1, 448) if block_dim == -1 else _log(rng, 64, 14336)
        rows = max(1, total // cols) if block_dim == -1 else 32 * max(1, total // cols // 32)
        return dict(kind=kind, op=op, rows=rows, cols=cols, block_dim=block_dim, fmt=rng.choice(_FMTS), dtype=dtype)
    return dict(kind=kind, op=op, count=_log(rng, 1 << 12, 5 << 23), fmt=rng.choice(_FMTS), dtype=dtype)


def _normal(g, *shape, dtype, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV).mul_(scale).to(dtype)


def _cast_values(g, n, dtype, sparse):
    """Heavy-tailed values, a thousandth of them zero, and where blocks are what counts a thousandth of the blocks all zero."""
    x = torch.randn(n, generator=g, device=DEV)
    chi2 = torch.zeros(n, device=DEV)
    for _ in range(3):
        chi2 += torch.randn(n, generator=g, device=DEV) ** 2
    x = x / (chi2 / 3.0).sqrt_() * 0.02
    few = torch.randint(0, n, (max(n // 1000, 1),), generator=g, device=DEV)
    x[few] *= 1.0e4
    x[torch.randint(0, n, (max(n // 1000, 1),), generator=g, device=DEV)] = 0.0
    if sparse:
        blocks = x[:n // 32 * 32].view(-1, 32)
        blocks[torch.randint(0, max(blocks.shape[0], 1), (blocks.shape[0] // 1000 + 1,), generator=g, device=DEV)] = 0.0
        x[int(torch.randint(0, n, (1,), generator=g, device=DEV))] = float("inf")
        x[int(torch.randint(0, n, (1,), generator=g, device=DEV))] = float("nan")
    return x.to(dtype)


def _mxfp_layer(weight, bias, case, layer):
    xq, wq = MXFP[case["x_fmt"]], MXFP[case["w_fmt"]]
    return MXFPLinearPTQ(weight=weight, bias=bias, x_mxfp_meta=xq if layer.startswith("Xq") else None, w_mxfp_meta=wq, b_mxfp_meta=None,
                         layer_type=layer, backend="fused")


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        dtype = getattr(torch, case["dtype"])
        small = case["family"] == "minifloat"      # element formats without a scale: weights of a size that the format holds
        w = _normal(g, case["n"], case["k"], dtype=dtype, scale=0.5 if small else 0.02)
        b = _normal(g, case["n"], dtype=dtype) if case["bias"] else None
        x = _normal(g, case["rows"], case["k"], dtype=dtype)
        if small:
            layer = MinifloatLinearPTQ(weight=w, bias=b, x_minifloat_meta=MINIFLOAT[case["x_fmt"]] if case["layer"].startswith("Xq") else None,
                                       w_minifloat_meta=MINIFLOAT[case["w_fmt"]], b_minifloat_meta=None, layer_type=case["layer"], backend="fused")
        else:
            layer = _mxfp_layer(w, b, case, case["layer"])
        return dict(kind=kind, x=x, layer=layer)
    if kind == "linear_call":
        w = _normal(g, case["n"], case["k"], dtype=torch.bfloat16, scale=0.02)
        scales, elements, meta = MX.extract_mxfp_components(w, block_dim=1, mxfp_meta=MXFP[case["w_fmt"]])
        return dict(kind=kind, x=_normal(g, case["rows"], case["k"], dtype=torch.bfloat16), x_meta=MXFP[case["x_fmt"]], w_scales=scales,
                    w_elements=elements, w_meta=meta)
    if kind == "mlp":
        gate_up = _mxfp_layer(_normal(g, 2 * case["inter"], case["hidden"], dtype=torch.bfloat16, scale=0.02), None, case, "XqWqB")
        down = _mxfp_layer(_normal(g, case["hidden"], case["inter"], dtype=torch.bfloat16, scale=0.02), None, case, "XqWqB")
        return dict(kind=kind, x=_normal(g, case["rows"], case["hidden"], dtype=torch.bfloat16), gate_up=gate_up, down=down)
    if kind == "matmul":
        b, h, q, s, d = case["batch"], case["heads"], case["q_len"], case["kv_len"], case["head_dim"]
        if case["product"] == "qk":
            left, right = _normal(g, b, h, q, d, dtype=torch.bfloat16), _normal(g, b, h, s, d, dtype=torch.bfloat16).transpose(-1, -2)
        else:
            left = torch.softmax(torch.randn(b, h, q, s, generator=g, device=DEV), dim=-1).to(torch.bfloat16)
            right = _normal(g, b, h, s, d, dtype=torch.bfloat16)
        return dict(kind=kind, left=left, right=right, meta=MXFP[case["fmt"]])
    dtype = getattr(torch, case["dtype"])
    if kind == "mxfp_cast":
        x = _cast_values(g, case["rows"] * case["cols"], dtype, True).view(case["rows"], case["cols"])
        return dict(kind=kind, op=case["op"], x=x, block_dim=case["block_dim"], meta=MXFP[case["fmt"]])
    return dict(kind=kind, op=case["op"], x=_cast_values(g, case["count"], dtype, False), meta=MINIFLOAT[case["fmt"]])


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "linear_call":
        return MX.mxfp_linear(x=state["x"], x_meta=state["x_meta"], w=None, w_scales=state["w_scales"], w_elements=state["w_elements"],
                              w_tensor_meta=state["w_meta"], b=None, b_scales=None, b_elements=None, b_tensor_meta=None, layer_type="XqWqB",
                              backend="fused")
    if kind == "mlp":
        gate, up = state["gate_up"](state["x"]).chunk(2, dim=-1)
        return state["down"].forward_swiglu(gate, up)
    if kind == "matmul":
        return MX.mxfp_matmul(state["left"], state["right"], state["meta"], state["meta"], "XqWq", "fused")
    if kind == "mxfp_cast":
        if state["op"] == "qdq":
            return MX.quantize_dequantize(state["x"], block_dim=state["block_dim"], mxfp_meta=state["meta"])
        scales, elements, meta = MX.extract_mxfp_components(state["x"], block_dim=state["block_dim"], mxfp_meta=state["meta"])
        return scales, elements, MX.compose_mxfp_tensor(scales, elements, meta)
    if state["op"] == "qdq":
        return MF.quantize_dequantize(state["x"], state["meta"])
    codes, meta = MF.extract_minifloat_component(state["x"], state["meta"])
    return codes.view(torch.int16), MF.compose_minifloat_component(codes, meta)   # (few tensor operations take uint16)


def work(case):
    """Codes are one byte each (two in the minifloat casts, which hand out uint16), block scales one byte per 32."""
    kind = case["kind"]
    if kind in ("linear", "linear_call"):
        m, k, n = case["rows"], case["k"], case["n"]
        size = SIZE[case.get("dtype", "bfloat16")]
        scaled = kind == "linear_call" or case["family"] == "mxfp"
        return {"bytes": m * k * size + n * k * (33 / 32 if scaled else 1) + m * n * size, "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 2 * m * h * 2 + 3 * h * i * 33 / 32, "flops": 2 * m * h * i * 3}
    if kind == "matmul":
        m, k, n = case["q_len"], case["head_dim"], case["kv_len"]
        if case["product"] == "pv":
            k, n = n, k
        return {"bytes": case["batch"] * case["heads"] * 2 * (m * k + k * n + m * n), "flops": case["batch"] * case["heads"] * 2 * m * n * k}
    size = SIZE[case["dtype"]]
    count = case["count"] if kind == "minifloat_cast" else case["rows"] * case["cols"]
    if case["op"] == "qdq":
        return {"bytes": 2 * count * size, "flops": 0}
    code = 2 if kind == "minifloat_cast" else 33 / 32
    # x in, codes out and in again, values out
    return {"bytes": 2 * count * size + 2 * count * code, "flops": 0}


def tolerance(case):
    """Casts are defined bit for bit.  A product's result is rounded to the output type after fp32 sums, whose order is free:
    a bf16 result then differs in a last bit here and there (up to 2.3e-4 in norm against the same product summed in float64:
    the matrix unit of the block-scaled products adds 32 products at a time with fewer bits than a chain of fp32 additions).
    In the SwiGLU block such a bit can move an element to the next FP8 code before the second product: 3e-3 measured.
    fp32 results of quantised fp32 operands: up to 6e-8."""
    kind = case["kind"]
    if kind.endswith("cast"):
        return "exact"
    if kind == "mlp":
        return {"rel": 1e-2}
    if case.get("dtype") == "float32":
        return {"rel": 4e-7}
    return {"rel": 1e-3}
