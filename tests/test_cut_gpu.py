"""Problems that a call cuts in two although the queries report one launch: plain, with rows of C at odd addresses, block-scaled."""
import pytest
import torch

import gemm_kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dt", [(1000, 50257, 768, torch.bfloat16), (3748, 13208, 640, torch.float16), (6784, 2504, 1792, torch.bfloat16),
                                      (1509, 11192, 3200, torch.float8_e4m3fn)])
def test_plain(M, N, K, dt):
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = (torch.randint(-2, 3, (r, K), generator=g, device="cuda", dtype=torch.float32) for r in (M, N))
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16 if dt == torch.float8_e4m3fn else dt, device="cuda")
    one = torch.ones(1, device="cuda")
    if dt == torch.float8_e4m3fn:
        gemm_kernels.gemm_tn_fp8(x.to(dt), w.to(dt), one, one, C)
    else:
        gemm_kernels.gemm_tn_test(x.to(dt), w.to(dt), C)
    assert torch.equal(C, (x @ w.T).to(C.dtype))      # sums of small integers are exact in fp32


@pytest.mark.parametrize("M,N,K", [(1509, 11192, 4864), (448, 34448, 1280), (2247, 8448, 3584)])
def test_block_scaled(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(2)
    x, w = (torch.randint(-2, 3, (r, K), generator=g, device="cuda", dtype=torch.float32) for r in (M, N))
    sx, sw = (torch.randint(126, 129, (r, K // 32), generator=g, device="cuda").to(torch.uint8) for r in (M, N))
    want = (x * torch.exp2(sx.float() - 127).repeat_interleave(32, 1)) @ (w * torch.exp2(sw.float() - 127).repeat_interleave(32, 1)).T
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    gemm_kernels.gemm_tn_mxfp8(x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), sx, sw, C)
    assert torch.equal(C, want.to(torch.bfloat16))


# pieces that run on other tiles than a plan with splits of K has, on the kernel for few outputs, or split in the room that the query asks for
@pytest.mark.parametrize("M,N,K,dt", [(565, 23296, 3712, torch.bfloat16), (4113, 8023, 880, torch.bfloat16), (3094, 16012, 4096, torch.float16),
                                      (2302, 22144, 2048, torch.float8_e4m3fn)])
def test_plain_pieces(M, N, K, dt):
    test_plain(M, N, K, dt)


@pytest.mark.parametrize("M,N,K", [(4143, 4096, 1920), (1480, 12160, 8320), (670, 23916, 2432), (3031, 6112, 7296)])
def test_block_scaled_pieces(M, N, K):
    test_block_scaled(M, N, K)
