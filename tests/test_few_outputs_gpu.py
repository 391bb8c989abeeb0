"""The kernel for products of few outputs, on operands of small integers: every sum is exact in fp32, so the result is the rounded
product to the bit.  What lies around C keeps its bits."""
import pytest
import torch

import gemm_kernels
from tests import abi_ctypes as ac
from tests.few_outputs_cases import ANY_ROWS, MX, PLAIN

pytestmark = pytest.mark.gpu
DT = {ac.BF16: torch.bfloat16, ac.F16: torch.float16, ac.E4M3: torch.float8_e4m3fn}


def integers(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randint(-3, 4, (M, K), generator=g, device="cuda", dtype=torch.float32)
    x *= torch.rand((M, K), generator=g, device="cuda") < min(1.0, 200 / K)      # fp16: sums stay below its largest value
    return x, torch.randint(-3, 4, (N, K), generator=g, device="cuda", dtype=torch.float32)


@pytest.mark.parametrize("M,N,K,code", PLAIN)
def test_plain(M, N, K, code):
    abi = ac.load()
    x, w = integers(M, N, K)
    A, B, want = x.to(DT[code]), w.to(DT[code]), x.double() @ w.double().T
    for out_code, out in ((ac.BF16, torch.bfloat16), (ac.F16, torch.float16)):
        for n, offset, pad in ((N, 0, 0), (N, 4, 8), (N, 1, 3), (N - 1, 0, 0), (N - 3, 1, 1)):
            if n < 1:
                continue
            ldc = n + pad
            buf = torch.full((M * ldc + 16,), 0x5a5a, dtype=torch.int16, device="cuda")
            C = torch.as_strided(buf, (M, n), (ldc, 1), offset)
            ws = torch.empty(1 << 24, dtype=torch.uint8, device="cuda")
            st = abi.mi355_gemm_tn(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, n, K, K, K, ldc, code, out_code, 1.0, ac.AUTO,
                                   ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
            assert st == ac.OK
            assert torch.equal(C.view(out), want[:, :n].to(torch.float32).to(out)), (n, offset, pad)
            C.fill_(0x5a5a)
            assert bool((buf == 0x5a5a).all()), (n, offset, pad)


@pytest.mark.parametrize("M,N,K", MX)
def test_block_scaled(M, N, K):
    x, w = integers(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(5)
    sx, sw = (torch.randint(125, 130, (r, K // 32), generator=g, device="cuda").to(torch.uint8) for r in (M, N))
    scaled = [v.double() * torch.exp2(s.double() - 127).repeat_interleave(32, 1) for v, s in ((x, sx), (w, sw))]
    want = scaled[0] @ scaled[1].T
    for out in (torch.bfloat16, torch.float16):
        C = torch.full((M, N), float("nan"), dtype=out, device="cuda")
        gemm_kernels.gemm_tn_mxfp8(x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), sx, sw, C)
        assert torch.equal(C, want.to(torch.float32).to(out))


@pytest.mark.parametrize("M,N,K,code,offset,gap", ANY_ROWS)
def test_rows_of_any_alignment(M, N, K, code, offset, gap):
    """What lies between the rows and around the operands is NaN."""
    abi = ac.load()
    x, w = integers(M, N, K)
    want = x.double() @ w.double().T
    views = []
    for v in (x, w):
        nan = torch.full((offset + v.shape[0] * (K + gap),), float("nan"), device="cuda").to(DT[code])
        view = torch.as_strided(nan, v.shape, (K + gap, 1), offset)
        view.copy_(v)
        views.append(view)
    A, B = views
    ws = torch.empty(1 << 27, dtype=torch.uint8, device="cuda")
    for pad in (0, 1, 2):
        C = torch.full((M, N + pad), float("nan"), dtype=torch.bfloat16, device="cuda")
        st = abi.mi355_gemm_tn(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K + gap, K + gap, N + pad, code, ac.BF16, 1.0, ac.AUTO,
                               ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
        assert st == ac.OK
        assert torch.equal(C[:, :N], want.to(torch.float32).to(torch.bfloat16)) and bool(C[:, N:].isnan().all())
