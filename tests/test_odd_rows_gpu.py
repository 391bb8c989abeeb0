"""Rows of C at every 2-byte alignment out of the tile kernels: each way an octet of columns can straddle a wave's, a tile's and
the matrix's last column.  Operands of small integers, so that every sum is exact in bf16; the rest of the buffer keeps its bits.
"""
import pytest
import torch

from tests import abi_ctypes as ac

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("tile", [256, 384, 128])     # 256 x 256, 256 x 128, 128 x 128
def test_every_end_of_a_row(monkeypatch, dt, tile):
    monkeypatch.setenv("MI355_RING_TILE", str(tile))
    abi = ac.load()
    M, K = 259, 1024 if dt == torch.float8_e4m3fn else 128     # enough products for fp8 to be multiplied on the matrix cores
    g = torch.Generator().manual_seed(11)
    x = torch.randint(-2, 3, (M, K), generator=g) * (torch.rand((M, K), generator=g) < 0.1)
    w = torch.randint(-1, 2, (400, K), generator=g)
    want = (x.double() @ w.double().T)
    assert float(want.abs().max()) <= 256
    A, B, want = x.to(torch.float32).to(dt).cuda(), w.to(torch.float32).to(dt).cuda(), want.cuda()
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    for N in [*range(257, 274), *range(311, 330), *range(375, 393)]:
        for offset, pad in ((0, 0), (1, 0), (1, 1), (2, 1), (0, 3)):
            ldc = N + pad
            buf = torch.full((M * ldc + 64,), 0x5a5a, dtype=torch.int16, device="cuda")
            C = torch.as_strided(buf, (M, N), (ldc, 1), offset)
            st = abi.mi355_gemm_tn(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, K, ldc, ac.torch_code(dt), ac.BF16, 1.0,
                                   ac.AUTO, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
            assert st == ac.OK
            assert torch.equal(C.view(torch.bfloat16).double(), want[:, :N]), (N, offset, pad)
            C.fill_(0x5a5a)
            assert bool((buf == 0x5a5a).all()), (N, offset, pad)
