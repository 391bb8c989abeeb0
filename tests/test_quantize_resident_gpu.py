"""The per-tensor quantiser on tensors that it reads once (80 to 128 MiB): the contract in torch ops, code for code, at scales that
the product with a reciprocal gets right and at such that it does not, with what is left to the kernel behind, and around the limits."""
import ctypes
import random

import pytest
import torch

import gemm_kernels
from gemm_kernels.quant import quantize_e4m3_torch
from tests import abi_ctypes as ac

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


@pytest.fixture
def masked_stream():
    """A stream on all compute units but one: not all workgroups can run at the same time on it."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    words = [0xffffffff] * (cus // 32) + [(1 << cus % 32) - 1] * (cus % 32 != 0)
    words[-1] >>= 1
    hip, handle = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(handle), len(words), (ctypes.c_uint32 * len(words))(*words)) == 0
    yield torch.cuda.ExternalStream(handle.value)
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0


def test_stream_with_a_mask(abi, masked_stream):
    """No longer than without scratch memory, the way that reads twice (it took five times as long while the workgroups that ran waited
    for those that could not); half as long again is the measurement's."""
    n = 64 * MIB
    x = torch.randn(n, device="cuda").bfloat16()
    q, scale = torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(2 + 512, device="cuda")
    want, want_scale = gemm_kernels.quantize_e4m3(x)
    abi.mi355_quantize_e4m3_scratch.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int64] + 3 * [ctypes.c_void_p] + [ctypes.c_size_t, ctypes.c_void_p]
    torch.cuda.synchronize()

    def us(scratch):
        times = []
        for _ in range(9):
            q.zero_()
            torch.cuda.synchronize()
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record(masked_stream)
            assert abi.mi355_quantize_e4m3_scratch(x.data_ptr(), ac.BF16, n, q.data_ptr(), scale.data_ptr(), scale.data_ptr() + 8 if scratch else None,
                                                   2048 if scratch else 0, masked_stream.cuda_stream) == ac.OK
            end.record(masked_stream)
            end.synchronize()
            times.append(begin.elapsed_time(end) * 1e3)
            assert float(scale[0]) == float(want_scale) and torch.equal(q, want.view(torch.uint8))
        return sorted(times)[4]

    assert us(True) < 1.5 * us(False)


def test_beside_other_work():
    """Two quantisers on two streams and a product on a third, whose workgroups take the compute units from one another."""
    streams = [torch.cuda.Stream() for _ in range(3)]
    xs = [torch.randn(64 * MIB, device="cuda").mul_(1 + i).bfloat16() for i in range(2)]
    want = [gemm_kernels.quantize_e4m3(x) for x in xs]
    a = torch.randint(-2, 3, (4352, 4096), device="cuda").bfloat16()
    c = torch.empty(4352, 4352, dtype=torch.bfloat16, device="cuda")
    product = (a.float() @ a.float().T).bfloat16()
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(4):
        with torch.cuda.stream(streams[2]):
            gemm_kernels.gemm_tn_test(a, a, c)
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got[i].append(gemm_kernels.quantize_e4m3(xs[i]))
    torch.cuda.synchronize()
    assert torch.equal(c, product)
    for i in range(2):
        for q, scale in got[i]:
            assert float(scale) == float(want[i][1]) and torch.equal(q.view(torch.uint8), want[i][0].view(torch.uint8))
