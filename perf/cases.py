"""Timed cases of the IntentIR execution backend: what is run, what it must move, and what it must give.

A program that uses this package lowers an IntentIR document once per shape, keeps the lowered kernel,
and launches it on device-resident tensors with ``launch_lowered``; a pass here is that one call.  The
documents are the workloads of ``intent_ir_amd/configs.py`` and the forms that the tests and the kernel
runner lower (row sums, element-wise chains, matmul with B given as [N, K]).  Host arrays in and out
(``run_lowered``) are bound by the copies over PCIe and are not timed.

``listed()`` spans the range: the reference's smoke shape, where a call is all latency, the benchmark
shapes, a decode step against a vocabulary, ragged rows and ragged products, f32, f16 and bf16.
``draw(rng)`` gives further sizes of the same kinds.
"""

from __future__ import annotations

import math

import torch

from intent_ir_amd import launch_lowered, lower_intent_to_hip_kernel
from intent_ir_amd.configs import (any_kernel_dim_ir, bias_gelu_axpy_ir, layer_norm_persistent_ir, matmul_bias_relu2d_ir,
                                   softmax_inner_ir)
from intent_ir_amd.runtime import tensor_shapes, torch_dtype

EPS = 1e-5
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
MIN_ELEMENTS, MAX_ELEMENTS = 1 << 13, 1 << 26     # of a drawn matrix: 32 KiB to 256 MiB in f32
MAX_FLOPS = {"bf16": 1 << 39, "f32": 1 << 35}


def listed():
    return [
        # The smallest call: the reference's own smoke test of its matmul, relu(A @ B + bias) in f32.
        # Nothing but latency: argument checks, one launch, a few wavefronts.
        {"name": "matmul_f32_32x48x16", "kind": "matmul", "dtype": "f32", "layout": "nn", "M": 32, "N": 48, "K": 16},
        # The five benchmark workloads.
        {"name": "any_8192x4096", "kind": "any", "M": 8192, "N": 4096},
        {"name": "softmax_16384x1024", "kind": "softmax", "M": 16384, "N": 1024},
        {"name": "layernorm_f16_8192x4096", "kind": "layernorm", "dtype": "f16", "M": 8192, "N": 4096},
        {"name": "gelu_bf16_32768x8192", "kind": "gelu", "M": 32768, "N": 8192},
        {"name": "matmul_bf16_8192", "kind": "matmul", "dtype": "bf16", "layout": "nn", "M": 8192, "N": 8192, "K": 8192},
        # Sampling over a vocabulary: few rows, each far longer than a workgroup holds.
        {"name": "softmax_64x128256", "kind": "softmax", "M": 64, "N": 128256},
        # Few long rows: a whole-tensor statistic such as a norm or a loss.
        {"name": "sum_64x1048576", "kind": "sum", "M": 64, "N": 1 << 20},
        # LayerNorm as the reference types it (f32), over rows that start at any 4-byte boundary.
        {"name": "layernorm_f32_8192x4099", "kind": "layernorm", "dtype": "f32", "M": 8192, "N": 4099},
        # A chain without a kernel of its own, with an operand read across its rows.
        {"name": "transpose_bias_f32_8192", "kind": "transpose_bias", "M": 8192, "N": 8192},
        # A decode step's projection: 32 rows against a linear layer's weight given as [N, K].
        {"name": "matmul_bf16_32x32000x4096", "kind": "matmul", "dtype": "bf16", "layout": "nt", "M": 32, "N": 32000,
         "K": 4096},
        # A ragged product: 1000 rows, a width whose rows cannot start 16-byte aligned.
        {"name": "matmul_bf16_1000x1001x4096", "kind": "matmul", "dtype": "bf16", "layout": "nn", "M": 1000, "N": 1001,
         "K": 4096},
    ]


# ----------------------------------------------------------------------------- further sizes

def _log_int(rng, lo, hi):
    """lo..hi, even over the logarithm; half of them as they fall (odd ones too), half on a multiple that a
    tuned size would have."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        step = 64 if v >= 256 else 8 if v >= 16 else 1
        v = v // step * step
    return min(max(v, lo), hi)


def _rows(rng, n_lo, n_hi):
    n = _log_int(rng, n_lo, n_hi)
    return {"M": _log_int(rng, max(1, MIN_ELEMENTS // n), max(1, MAX_ELEMENTS // n)), "N": n}


def draw(rng):
    kind = rng.choice(["any", "sum", "softmax", "layernorm", "layernorm", "gelu", "bias_relu", "sigmoid",
                       "transpose_bias", "matmul", "matmul", "matmul", "matmul"])
    if kind == "layernorm":
        return {"kind": kind, "dtype": rng.choice(["f16", "f32"]), **_rows(rng, 32, 32768)}
    if kind == "softmax":
        return {"kind": kind, **_rows(rng, 16, 262144)}
    if kind in ("any", "sum"):
        return {"kind": kind, **_rows(rng, 16, 1 << 20)}
    if kind == "matmul":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        m = _log_int(rng, 1, 8192)       # 1 row of a decode step to a batch of prompts
        k = _log_int(rng, 16, 16384)
        n = _log_int(rng, 64, min(65536, max(64, MAX_FLOPS[dtype] // (2 * m * k)), MAX_ELEMENTS * 4 // k))
        return {"kind": kind, "dtype": dtype, "layout": rng.choice(["nn", "nt"]), "M": m, "N": n, "K": k}
    return {"kind": kind, **_rows(rng, 16, 32768)}


# ----------------------------------------------------------------------------- documents and inputs

def _t(dtype, *shape):
    return {"dtype": dtype, "shape": list(shape)}


def _op(name, inputs, output, **attrs):
    return {"op": name, "inputs": list(inputs), "output": output, "attrs": attrs}


def _ir(case):
    kind = case["kind"]
    if kind == "any":
        return any_kernel_dim_ir()
    if kind == "softmax":
        return softmax_inner_ir()
    if kind == "layernorm":
        return layer_norm_persistent_ir(case["dtype"])
    if kind == "gelu":
        return bias_gelu_axpy_ir()
    if kind == "matmul":
        ir = matmul_bias_relu2d_ir(case["dtype"])
        if case["layout"] == "nt":
            ir["tensors"]["B"] = _t(case["dtype"], "N", "K")
            ir["ops"][0]["attrs"] = {"transpose_b": True}
        return ir
    if kind == "sum":
        return {"name": "row_sum", "tensors": {"x": _t("f32", "M", "N"), "out": _t("f32", "M")},
                "ops": [_op("reduce_sum", ["x"], "out", dims=[1])], "outputs": ["out"]}
    if kind == "bias_relu":
        return {"name": "bias_relu", "outputs": ["y"],
                "tensors": {"x": _t("f32", "M", "N"), "b": _t("f32", "N"), "t": _t("f32", "M", "N"),
                            "y": _t("f32", "M", "N")},
                "ops": [_op("add", ["x", "b"], "t"), _op("relu", ["t"], "y")]}
    if kind == "transpose_bias":
        return {"name": "transpose_bias", "outputs": ["y"],
                "tensors": {"x": _t("f32", "N", "M"), "b": _t("f32", "N"), "xt": _t("f32", "M", "N"),
                            "y": _t("f32", "M", "N")},
                "ops": [_op("transpose", ["x"], "xt", perm=[1, 0]), _op("add", ["xt", "b"], "y")]}
    if kind == "sigmoid":
        return {"name": "sigmoid", "outputs": ["y"],
                "tensors": {"x": _t("bf16", "M", "N"), "u": _t("f32", "M", "N"), "e": _t("f32", "M", "N"),
                            "one": _t("f32"), "d": _t("f32", "M", "N"), "y": _t("bf16", "M", "N")},
                "ops": [_op("mul", ["x"], "u", mul_factor=-1.0), _op("exp", ["u"], "e"),
                        _op("const", [], "one", value=1.0, dtype="f32"), _op("add", ["e", "one"], "d"),
                        _op("div", ["one", "d"], "y")]}
    raise ValueError(kind)


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    kind, M, N = case["kind"], case["M"], case["N"]
    if kind == "any":           # sparse flags: most rows hold few non-zeros, many none
        x = randn(M, N)
        keep = torch.rand((M, N), generator=g, device="cuda") < 1.0 / (2 * N)
        return {"inp": torch.where(keep, x, torch.zeros((), device="cuda"))}
    if kind == "sum":           # non-negative terms (squares, losses, counts)
        return {"x": torch.rand((M, N), generator=g, device="cuda")}
    if kind == "softmax":       # logits, 1% of them far out
        x = randn(M, N) * 2.0
        far = torch.rand((M, N), generator=g, device="cuda") < 0.01
        return {"input_ptr": torch.where(far, torch.sign(x) * 30.0, x)}
    if kind == "layernorm":     # activations with a mean of their own
        dt = torch_dtype(case["dtype"])
        return {"in_ptr": (randn(M, N) + 0.25).to(dt), "weight_ptr": (1.0 + 0.1 * randn(N)).to(dt),
                "bias_ptr": (0.1 * randn(N)).to(dt)}
    if kind == "gelu":
        return {"x": randn(M, N).bfloat16(), "bias": (0.02 * randn(N)).bfloat16()}
    if kind == "bias_relu":
        return {"x": randn(M, N), "b": 0.1 * randn(N)}
    if kind == "transpose_bias":
        return {"x": randn(N, M), "b": 0.1 * randn(N)}
    if kind == "sigmoid":
        return {"x": (3.0 * randn(M, N)).bfloat16()}
    K, dt = case["K"], torch_dtype(case["dtype"])
    b = (N, K) if case["layout"] == "nt" else (K, N)
    return {"A": randn(M, K).to(dt), "B": (randn(*b) / math.sqrt(K)).to(dt), "bias": 0.1 * randn(N)}


# ----------------------------------------------------------------------------- one pass

def prepare(case, seed):
    bindings = {k: case[k] for k in ("M", "N", "K") if k in case}
    kernel = lower_intent_to_hip_kernel(_ir(case), shape_bindings=bindings)
    buffers = _inputs(case, seed)
    shapes = tensor_shapes(kernel.io_spec, kernel.bindings)
    for name in kernel.output_names:
        dt = torch_dtype(kernel.io_spec["tensors"][name]["dtype"])
        buffers[name] = torch.empty(shapes[name], dtype=dt, device="cuda")
    return {"kernel": kernel, "buffers": buffers}


def run(state):
    kernel, buffers = state["kernel"], state["buffers"]
    launch_lowered(kernel, buffers)
    return {name: buffers[name] for name in kernel.output_names}


def work(case):
    """Every input read once, every output written once; multiply-adds of the products, and for the other
    kinds the arithmetic per element of their formula."""
    kind, M, N = case["kind"], case["M"], case["N"]
    if kind == "any":
        return {"bytes": 4 * M * N + M, "flops": M * N}
    if kind == "sum":
        return {"bytes": 4 * M * N + 4 * M, "flops": M * N}
    if kind == "softmax":
        return {"bytes": 8 * M * N, "flops": 5 * M * N}
    if kind == "layernorm":
        e = BYTES[case["dtype"]]
        return {"bytes": 2 * e * M * N + 2 * e * N + 8 * M, "flops": 8 * M * N}
    if kind == "gelu":
        return {"bytes": 4 * M * N + 2 * N, "flops": 11 * M * N}
    if kind in ("bias_relu", "transpose_bias"):
        return {"bytes": 8 * M * N + 4 * N, "flops": 2 * M * N if kind == "bias_relu" else M * N}
    if kind == "sigmoid":
        return {"bytes": 4 * M * N, "flops": 4 * M * N}
    K, e = case["K"], BYTES[case["dtype"]]
    return {"bytes": e * (M * K + K * N + M * N) + 4 * N, "flops": 2 * M * N * K}


def tolerance(case):
    """About four times the distance from 64 bits that these kernels show (exact(), on the listed cases and
    a hundred drawn ones): the rounding of the output type for 16-bit outputs, the order of the sums and
    the last places of exp and rsqrt for 32-bit ones."""
    kind = case["kind"]
    if kind == "any":
        return "exact"
    if kind in ("gelu", "sigmoid") or (kind == "matmul" and case["dtype"] == "bf16"):
        return {"rel": 7e-3, "max": 2e-2}
    if kind == "layernorm" and case["dtype"] == "f16":
        return {"rel": 1e-3, "max": 4e-3}
    if kind == "matmul":
        return {"rel": 6e-6, "max": 4e-5}
    if kind in ("bias_relu", "transpose_bias"):
        return {"rel": 2e-7, "max": 5e-7}
    return {"rel": 1e-6, "max": 4e-6}


# ----------------------------------------------------------------------------- the same in 64 bits

def exact(case, seed):
    kind, M = case["kind"], case["M"]
    x = _inputs(case, seed)
    if kind == "any":
        return {"out": (x["inp"] != 0).any(dim=1)}
    if kind == "sum":
        return {"out": x["x"].double().sum(dim=1)}
    if kind == "softmax":
        return {"output_ptr": torch.softmax(x["input_ptr"].double(), dim=1)}
    if kind == "layernorm":
        v = x["in_ptr"].double()
        mean = v.mean(dim=1, keepdim=True)
        d = v - mean
        rstd = 1.0 / torch.sqrt((d * d).mean(dim=1, keepdim=True) + EPS)
        return {"out_ptr": d * rstd * x["weight_ptr"].double() + x["bias_ptr"].double(),
                "out_mean_ptr": mean.reshape(M), "out_rstd_ptr": rstd.reshape(M)}
    if kind == "gelu":
        v = x["x"].double()
        z = v + x["bias"].double()
        return {"y": torch.nn.functional.gelu(z, approximate="tanh") * 0.5 + v}
    if kind == "bias_relu":
        return {"y": torch.relu(x["x"].double() + x["b"].double())}
    if kind == "transpose_bias":
        return {"y": x["x"].double().t() + x["b"].double()}
    if kind == "sigmoid":
        return {"y": torch.sigmoid(x["x"].double())}
    b = x["B"].double()
    if case["layout"] == "nt":
        b = b.t().contiguous()
    return {"C": torch.relu(x["A"].double() @ b + x["bias"].double())}
