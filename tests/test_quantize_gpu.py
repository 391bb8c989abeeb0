"""Per-tensor fp8 quantiser on the device at the edges of its launch rules and of its division.

Expected codes: torch's fp32 division on the CPU (correctly rounded) and its e4m3fn cast, both restated in
gemm_kernels.quant.quantize_e4m3_torch.  Codes and scales are compared bit for bit.
"""
import pytest
import torch

from tests import abi_ctypes as ac

pytestmark = pytest.mark.gpu


def expected(x):
    from gemm_kernels.quant import quantize_e4m3_torch
    q, s = quantize_e4m3_torch(x)
    return q.view(torch.uint8), float(s)


# One workgroup of the single launch, its last one, the first two-launch sizes, remainders of a run and of a group of eight.
@pytest.mark.parametrize("dtype,n", [
    (torch.bfloat16, 1), (torch.bfloat16, 8191), (torch.bfloat16, 131072), (torch.bfloat16, 131073), (torch.bfloat16, 8192 * 17 + 2055),
    (torch.float16, 131072 + 8), (torch.float32, 65536), (torch.float32, 65537), (torch.float32, 3 * 8192 - 1),
    (torch.bfloat16, (32 << 20) + 8 * 257 + 3)])
def test_sizes_around_the_launch_rules(dtype, n):
    import gemm_kernels
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(dtype)
    want_q, want_s = expected(x)
    for _ in range(2):
        q, s = gemm_kernels.quantize_e4m3(x.cuda())
        assert float(s) == want_s
        assert torch.equal(q.cpu().view(torch.uint8), want_q)


# Around 32 MiB of input (1024 workgroups up to there) with more than one turn of four pieces each, and with pieces left over.
@pytest.mark.parametrize("dtype,n", [
    (torch.bfloat16, 16 << 20), (torch.bfloat16, (16 << 20) + 5), (torch.float16, 4099 * 2048 + 9), (torch.float32, 8 << 20),
    (torch.float32, (8 << 20) + 2055), (torch.bfloat16, 1023 * 2048 + 8), (torch.bfloat16, 4096 * 2048 - 8)])
def test_pieces_of_a_workgroup(dtype, n):
    import gemm_kernels
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(dtype)
    want_q, want_s = expected(x)
    q, s = gemm_kernels.quantize_e4m3(x.cuda())
    assert float(s) == want_s
    assert torch.equal(q.cpu().view(torch.uint8), want_q)


# amax from the subnormals to the largest finite number: the corrected reciprocal up to and beyond its range, the division outside.
# The smallest is above 448 * 2^-150: below, the scale itself is 0 and the quotients are infinities and NaNs of either sign.
@pytest.mark.parametrize("amax", [1e-42, 3e-39, 448 * 2.0 ** -61, 448 * 2.0 ** -60, 448 * 2.0 ** -59, 7e-6, 0.7, 300.0, 448 * 1.99999988,
                                  448 * 2.0 ** 99, 448 * 2.0 ** 101, 3.4028234663852886e38])
@pytest.mark.parametrize("n", [60000, 200000])
def test_quotients_for_every_size_of_scale(amax, n):
    import gemm_kernels
    g = torch.Generator().manual_seed(int(n))
    x = (torch.rand(n, generator=g, dtype=torch.float64) * 2 - 1) * torch.exp2(-22 * torch.rand(n, generator=g, dtype=torch.float64))
    x = (x * amax).clamp(-amax, amax).float()
    x[0], x[1], x[2] = torch.tensor(amax, dtype=torch.float64).float(), 0.0, -0.0
    want_q, want_s = expected(x)
    q, s = gemm_kernels.quantize_e4m3(x.cuda())
    assert float(s) == want_s
    assert torch.equal(q.cpu().view(torch.uint8), want_q)


@pytest.mark.parametrize("n", [4096, 300000])
def test_every_bf16_pattern_infinities_and_nan(n):
    """Every finite bf16 value at once; then with an infinity (every number becomes 0) and NaNs (code 0x7f, ignored by amax)."""
    import gemm_kernels
    bits = torch.arange(0, 65536, dtype=torch.int32).to(torch.int16)
    every = bits.view(torch.bfloat16)
    every = every[torch.isfinite(every.float())]
    x = torch.cat([every, torch.randn(n, generator=torch.Generator().manual_seed(1)).bfloat16()])
    want_q, want_s = expected(x)
    q, s = gemm_kernels.quantize_e4m3(x.cuda())
    assert float(s) == want_s and torch.equal(q.cpu().view(torch.uint8), want_q)

    y = torch.randn(n, generator=torch.Generator().manual_seed(n)).bfloat16()
    y[3] = y[n - 1] = 0
    want_q, want_s = expected(y)
    y[3], y[n - 1] = float("nan"), -float("nan")
    q, s = gemm_kernels.quantize_e4m3(y.cuda())
    got = q.cpu().view(torch.uint8)
    assert int(got[3]) == 0x7f and int(got[n - 1]) == 0x7f
    keep = torch.ones(n, dtype=torch.bool)
    keep[3] = keep[n - 1] = False
    assert float(s) == want_s
    assert torch.equal(got[keep], want_q[keep])

    y[5] = float("inf")
    q, s = gemm_kernels.quantize_e4m3(y.cuda())
    got = q.cpu().view(torch.uint8)
    assert float(s) == float("inf") and int(got[5]) & 0x7f == 0x7f
    keep[5] = False
    assert not (got[keep] & 0x7f).any()


@pytest.mark.parametrize("n", [1000, 131073, 1 << 20])
def test_with_and_without_scratch_memory(n):
    """The entry point that has no scratch memory, and one with room for three maxima only, give the same bytes."""
    L = ac.load()
    import ctypes
    L.mi355_quantize_e4m3_scratch.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p,
                                              ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
    L.mi355_quantize_e4m3_scratch_bytes.restype = ctypes.c_size_t
    L.mi355_quantize_e4m3_scratch_bytes.argtypes = [ctypes.c_int64]
    x = torch.randn(n, generator=torch.Generator().manual_seed(1)).bfloat16()
    want_q, want_s = expected(x)
    xd, stream = x.cuda(), torch.cuda.current_stream().cuda_stream
    room = L.mi355_quantize_e4m3_scratch_bytes(n)
    for scratch_bytes in (None, 12, room):
        q, sa = torch.zeros(n, dtype=torch.uint8, device="cuda"), torch.zeros(2, device="cuda")
        scratch = torch.full((max(room, 64),), 255, dtype=torch.uint8, device="cuda")
        if scratch_bytes is None:
            st = L.mi355_quantize_e4m3(xd.data_ptr(), ac.BF16, n, q.data_ptr(), sa.data_ptr(), stream)
        else:
            st = L.mi355_quantize_e4m3_scratch(xd.data_ptr(), ac.BF16, n, q.data_ptr(), sa.data_ptr(), scratch.data_ptr(),
                                               scratch_bytes, stream)
        assert st == ac.OK
        assert float(sa[0]) == want_s and float(sa[1]) == float(x.float().abs().max())
        assert torch.equal(q.cpu(), want_q)
