"""The per-tensor quantiser on tensors that it reads once (80 to 128 MiB): the contract in torch ops, code for code, at scales that
the product with a reciprocal gets right and at such that it does not, with what is left to the kernel behind, and around the limits."""
import random

import pytest
import torch

import gemm_kernels
from gemm_kernels.quant import quantize_e4m3_torch

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def check(x):
    q, scale = gemm_kernels.quantize_e4m3(x)
    nan = torch.isnan(x)
    want, want_scale = quantize_e4m3_torch(torch.where(nan, torch.zeros_like(x), x))
    nan |= torch.isinf(x)      # infinity over the infinite scale
    want = torch.where(nan, torch.full_like(want.view(torch.uint8), 0x7f), want.view(torch.uint8))
    assert float(scale) == float(want_scale)
    assert torch.equal(q.view(torch.uint8), want)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_every_value_at_many_scales(dt):
    rng = random.Random(5)
    values = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dt)
    values = values[torch.isfinite(values.float())]
    for i in range(40):
        amax = float(torch.tensor(2 ** (rng.uniform(-10, 15) if dt == torch.float16 else rng.uniform(-70, 110))).to(dt))
        v = values[values.float().abs() <= amax]
        n = 81 * MIB // 2 + rng.randint(0, 5000)
        x = v.repeat(n // v.numel() + 1)[:n]
        x[rng.randint(0, n - 1)] = -amax
        if i % 8 == 7:
            x[rng.randint(0, n - 1)] = float("nan")
        check(x)


@pytest.mark.parametrize("wait", [None, "0"])
@pytest.mark.parametrize("dt,n", [(torch.bfloat16, 40 * MIB - 1), (torch.bfloat16, 40 * MIB), (torch.float16, 50 * MIB + 4095), (torch.bfloat16, 64 * MIB),
                                  (torch.bfloat16, 64 * MIB + 4095), (torch.bfloat16, 64 * MIB + 4096), (torch.float32, 20 * MIB + 3),
                                  (torch.float32, 32 * MIB + 2047), (torch.float32, 32 * MIB + 2048)])
def test_limits(monkeypatch, dt, n, wait):
    if wait is not None:
        monkeypatch.setenv("MI355_QUANTIZE_WAIT_US", wait)
    g = torch.Generator(device="cuda").manual_seed(n % 1000)
    x = torch.randn(n, generator=g, device="cuda").to(dt)
    x[-1] = 9.0      # the largest is the last
    check(x)
    x[7] = float("inf")
    check(x)


def test_graph():
    x = torch.randn(48 * MIB, device="cuda").bfloat16()
    gemm_kernels.quantize_e4m3(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q, scale = gemm_kernels.quantize_e4m3(x)
    for i in range(4):
        x.copy_(torch.randn(48 * MIB, device="cuda").mul_(1 + i))
        graph.replay()
        torch.cuda.synchronize()
        want, want_scale = gemm_kernels.quantize_e4m3(x)
        assert float(scale) == float(want_scale) and torch.equal(q.view(torch.uint8), want.view(torch.uint8))
