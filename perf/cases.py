"""Timed cases of the library: the calls its users make, through the public Python entry points.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights and output buffer of one caller, on the GPU
    run(state)          one pass through the entry points
    work(case)          bytes and operations a pass cannot do without
    tolerance(case)     how far two correct results may lie apart

A case is one of four operations ("op"):

    gemm       gemm_tn_test(A, B, C): 16-bit operands and output
    fp8        a linear layer with per-tensor fp8: the activations are quantised by the call
               (quantize_e4m3) and multiplied (gemm_tn_fp8) with weights that were quantised once
    mx         the same with OCP MX block scales (quantize_mxfp8, gemm_tn_mxfp8), weight scales
               kept in the layout the GEMM reads
    quant_e4m3, quant_mx   a tensor quantised on its own, as weights are when a model is loaded

M is the number of tokens (rows of the activations), N the output features, K the input features.
"""
import math
import os
import sys

import torch

# The package folder is not an importable name itself; the caller's working folder is the repository's root.
sys.path.insert(0, os.path.join(os.getcwd(), "cute-examples_amd"))
import gemm_kernels  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

LARGEST = 8192 ** 3   # M * N * K of the largest listed product
LARGEST_QUANT = 8192 * 14336


def listed():
    return [
        # The smallest product of the benchmark configurations: launch latency.
        {"name": "fp16_512", "op": "gemm", "M": 512, "N": 512, "K": 512, "dtype": "fp16", "dist": "inv_sqrt_k"},
        # One decode step of a few sequences: an up projection in bf16, reading the weights once.
        {"name": "bf16_decode_16", "op": "gemm", "M": 16, "N": 14336, "K": 4096, "dtype": "bf16", "dist": "weights"},
        # The same step of an fp8 model: the attention input projection, with its activations quantised on the way.
        {"name": "fp8_decode_16", "op": "fp8", "M": 16, "N": 6144, "K": 4096, "dtype": "bf16", "dist": "weights"},
        # A larger decode batch of a block-scaled model: the down projection (long K).
        {"name": "mx_decode_64", "op": "mx", "M": 64, "N": 4096, "K": 14336, "dtype": "bf16", "dist": "weights"},
        # A few hundred tokens at once (speculative or batched decoding): weights and matrix cores both count.
        {"name": "bf16_batch_256", "op": "gemm", "M": 256, "N": 14336, "K": 4096, "dtype": "bf16", "dist": "weights"},
        # Everything ragged, no row aligned: half precision with an odd number of rows.
        {"name": "fp16_ragged", "op": "gemm", "M": 515, "N": 2050, "K": 4100, "dtype": "fp16", "dist": "inv_sqrt_k"},
        # Logits over an odd-sized vocabulary: a short K and an output far larger than the inputs.
        {"name": "bf16_vocabulary", "op": "gemm", "M": 1000, "N": 50257, "K": 768, "dtype": "bf16", "dist": "weights"},
        # Prefill of a block-scaled model: up projection of two thousand tokens.
        {"name": "mx_prefill_2048", "op": "mx", "M": 2048, "N": 14336, "K": 4096, "dtype": "bf16", "dist": "weights"},
        # The ordinary square product of the benchmark configurations.
        {"name": "bf16_4096", "op": "gemm", "M": 4096, "N": 4096, "K": 4096, "dtype": "bf16", "dist": "uniform"},
        # Weights quantised per tensor when a model is loaded.
        {"name": "quant_e4m3_8192", "op": "quant_e4m3", "M": 8192, "N": 0, "K": 8192, "dtype": "bf16", "dist": "normal"},
        # The large fp8 product of the headline metric, as a layer: the activations are quantised on the way.
        {"name": "fp8_prefill_8192", "op": "fp8", "M": 8192, "N": 8192, "K": 8192, "dtype": "bf16", "dist": "normal"},
        # The headline product.
        {"name": "bf16_8192", "op": "gemm", "M": 8192, "N": 8192, "K": 8192, "dtype": "bf16", "dist": "normal"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemm"] * 5 + ["fp8"] * 2 + ["mx"] * 2 + ["quant_e4m3", "quant_mx"])
    if op.startswith("quant"):
        while True:
            M, K = _log_uniform(rng, 1, 16384), _log_uniform(rng, 128, 16384)
            if op == "quant_mx" or rng.random() < 0.6:
                K = (K + 127) // 128 * 128
            if M * K <= LARGEST_QUANT:
                return {"op": op, "M": M, "N": 0, "K": K, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "dist": "normal"}
    while True:
        M, N, K = _log_uniform(rng, 1, 8192), _log_uniform(rng, 128, 50257), _log_uniform(rng, 128, 14336)
        # Feature counts: mostly multiples of 128, sometimes of 16, sometimes anything (block scales take whole blocks).
        form = rng.random()
        step_n, step_k = (128, 128) if form < 0.6 else (16, 16) if form < 0.8 else (1, 1)
        if op == "mx":
            step_n, step_k = max(step_n, 4), 128
        N, K = (N + step_n - 1) // step_n * step_n, (K + step_k - 1) // step_k * step_k
        if M * N * K <= LARGEST:
            break
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    return {"op": op, "M": M, "N": N, "K": K, "dtype": dtype, "dist": rng.choice(["weights", "normal", "uniform"])}


def _operand(shape, case, role, generator):
    """Activations (role 0) or weights (role 1) with the distribution the case names."""
    dist = case["dist"]
    if dist == "uniform":
        x = torch.rand(shape, generator=generator, device="cuda", dtype=torch.float32).mul_(2.0).sub_(1.0)
    else:
        x = torch.randn(shape, generator=generator, device="cuda", dtype=torch.float32)
        if dist == "weights" and role == 1:
            x.mul_(0.02)
        elif dist == "inv_sqrt_k":
            x.mul_(case["K"] ** -0.5)
    return x.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, M, N, K = case["op"], case["M"], case["N"], case["K"]
    state = {"op": op, "x": _operand((M, K), case, 0, g)}
    if op.startswith("quant"):
        return state
    w = _operand((N, K), case, 1, g)
    state["c"] = torch.empty((M, N), device="cuda", dtype=DTYPES[case["dtype"]])
    if op == "gemm":
        state["w"] = w
    elif op == "fp8":
        state["w"], state["w_scale"] = gemm_kernels.quantize_e4m3(w)
    else:
        state["w"], state["w_scale"] = gemm_kernels.quantize_mxfp8(w, shuffled=True)
    return state


def run(state):
    op = state["op"]
    if op == "gemm":
        return gemm_kernels.gemm_tn_test(state["x"], state["w"], state["c"])
    if op == "fp8":
        x_q, x_scale = gemm_kernels.quantize_e4m3(state["x"])
        return gemm_kernels.gemm_tn_fp8(x_q, state["w"], x_scale, state["w_scale"], state["c"])
    if op == "mx":
        x_q, x_scale = gemm_kernels.quantize_mxfp8(state["x"], shuffled=True)
        return gemm_kernels.gemm_tn_mxfp8(x_q, state["w"], x_scale, state["w_scale"], state["c"], scales_shuffled=True)
    if op == "quant_e4m3":
        return gemm_kernels.quantize_e4m3(state["x"])
    return gemm_kernels.quantize_mxfp8(state["x"])


def work(case):
    op, M, N, K, es = case["op"], case["M"], case["N"], case["K"], BYTES[case["dtype"]]
    x = M * K * es
    if op == "quant_e4m3":
        return {"bytes": x + M * K + 4, "flops": 2 * M * K}          # a maximum and a division per element
    if op == "quant_mx":
        return {"bytes": x + M * K + M * K // 32, "flops": 2 * M * K}
    weights = {"gemm": N * K * es, "fp8": N * K, "mx": N * K + N * K // 32}[op]
    return {"bytes": x + weights + M * N * es, "flops": 2 * M * N * K}


def tolerance(case):
    """Four times the distance of this library's results from the products of the same (quantised) operands in 64 bits,
    rounded once to the output type (largest seen over 21 sizes: 5.0e-5 / 1.6e-5 for bf16 / fp16 operands, 2.3e-4 /
    8.1e-5 where the matrix cores add fp8 products).  All of that is results that round the other way by one unit, so
    outputs of few values get two such units on top; a single value may be two units off."""
    if case["op"].startswith("quant"):
        return "exact"                                                # codes and scales are fixed by the formats
    bf16 = case["dtype"] == "bf16"
    if case["op"] == "gemm":
        rel = 2e-4 if bf16 else 6.4e-5
    else:
        rel = 9.2e-4 if bf16 else 3.3e-4
    unit = 2.0 ** -7 if bf16 else 2.0 ** -10                          # largest unit in the last place over the value
    return {"rel": rel + unit * math.sqrt(2.0 / (case["M"] * case["N"])), "max": 2 * unit}
