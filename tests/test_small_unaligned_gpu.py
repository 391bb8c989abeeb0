"""Small products with rows of any alignment (gemm_tn_small.hip through MI355_VARIANT_AUTO; the generic kernel below K = 128).

Reference: the product in float64 on the CPU.  fp32 sums of exact products in any order are off by at most about
K * 2^-24 of the sum of magnitudes; the output's rounding (2^-8 bf16, 2^-11 fp16 of the value) comes on top.
"""
import pytest
import torch

from tests import abi_ctypes as ac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11), (torch.float8_e4m3fn, 2.0 ** -8)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 5, 9), (3, 4, 511), (4, 129, 513), (5, 7, 1023), (16, 1001, 1025), (17, 130, 2049),
                                   (1, 3000, 14335), (129, 33, 4099), (1000, 51, 257), (2, 2, 65)])
def test_against_float64(dt, ulp, M, N, K):
    abi = ac.load()
    g = torch.Generator().manual_seed(M + N + K)
    A, B = (torch.randn((r, K), generator=g).to(dt) for r in (M, N))
    out_dt = torch.bfloat16 if dt == torch.float8_e4m3fn else dt
    ldc, offset = N + 1, 1
    buf = torch.full((M * ldc + 8,), 0x5a5a, dtype=torch.int16, device="cuda")
    C = torch.as_strided(buf, (M, N), (ldc, 1), offset).view(out_dt)
    # operands end exactly where their storage ends, one element off 16-byte alignment
    Ad, Bd = (torch.cat([torch.zeros(1, dtype=torch.uint8 if dt == torch.float8_e4m3fn else torch.int16),
                         x.flatten().view(torch.uint8 if dt == torch.float8_e4m3fn else torch.int16)]).cuda()[1:] for x in (A, B))
    st = abi.mi355_gemm_tn(Ad.data_ptr(), Bd.data_ptr(), C.data_ptr(), M, N, K, K, K, ldc, ac.torch_code(dt), ac.torch_code(out_dt), 0.5,
                           ac.AUTO, None, 0, torch.cuda.current_stream().cuda_stream)
    assert st == ac.OK
    torch.cuda.synchronize()
    got = C.cpu().double()
    want = 0.5 * (A.double() @ B.double().T)
    bound = ulp * want.abs() + K * 2.0 ** -24 * 0.5 * (A.double().abs() @ B.double().abs().T) + 1e-7
    assert bool(((got - want).abs() <= bound).all())
    C.view(torch.int16).fill_(0x5a5a)
    assert bool((buf == 0x5a5a).all())
    assert float(A.double().abs().max()) < 448
    # infinities and NaN travel as in the products
    if K > 1 and dt != torch.float8_e4m3fn:
        A[0, K - 1] = float("inf")
        B[0, K - 1] = 0.0
        st = ac.gemm_tn(abi, A.cuda(), B.cuda(), C, 1.0, ac.AUTO)
        assert st == ac.OK and bool(torch.isnan(C[0, 0]))


@pytest.mark.parametrize("M,N,K", [(16, 33, 128), (16, 33, 1024), (5, 129, 4096), (17, 66, 14336)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
def test_sums_that_cancel_keep_32_bits(dt, M, N, K):
    """Only the rows of C are unaligned.  B's second half is the first one negated but for a few elements, so the sums are far
    smaller than what is added up.  Rounding to fp16 is off by at most 2^-11 of a value: 2^-11 / sqrt(3) in the norm if errors
    spread evenly up to that; fp32 sums add a few per cent of it."""
    abi = ac.load()
    g = torch.Generator().manual_seed(K)
    a, b = torch.randn(M, K // 2, generator=g).to(dt).float(), torch.randn(N, K // 2, generator=g).to(dt).float()
    A, B = torch.cat([a, a], 1), torch.cat([b, -b.scatter(1, torch.randint(0, K // 2, (N, 4), generator=g), 0.0)], 1)
    order = torch.randperm(K, generator=g)
    A, B = A[:, order].to(dt).contiguous(), B[:, order].to(dt).contiguous()
    want = A.double() @ B.double().T
    C = torch.zeros((M, N), dtype=torch.float16, device="cuda")
    assert ac.gemm_tn(abi, A.cuda(), B.cuda(), C) == ac.OK
    assert float((C.cpu().double() - want).norm() / want.norm()) <= 2.0 ** -11 / 3 ** 0.5
