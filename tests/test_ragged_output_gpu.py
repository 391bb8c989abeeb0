"""Outputs whose rows only their element type aligns (N or ldc not a multiple of 4, C at any 2-byte address), stored by the
matrix-core kernels directly, on every plan that can take them; and operands repacked for an unaligned K.

The reference product is torch's in float64 on the CPU; tolerances are those of the other GPU tests (1e-2 for 16-bit
operands, 3e-2 for fp8, relative Frobenius).  Everything around C must keep its bits.
"""
import ctypes

import pytest
import torch

from tests import abi_ctypes as ac

pytestmark = pytest.mark.gpu
OUT = {torch.bfloat16: torch.bfloat16, torch.float16: torch.float16, torch.float8_e4m3fn: torch.bfloat16}


def operand(rows, K, dt, seed):
    x = torch.randn((rows, K), generator=torch.Generator().manual_seed(seed))
    return (x.clamp_(-30, 30) if dt == torch.float8_e4m3fn else x).to(dt)


@pytest.fixture(scope="module")
def abi():
    return ac.load()


def run(abi, A, B, offset, ldc, workspace=True, room=True, ws_bytes=None):
    """C inside a buffer of a known pattern, `offset` elements in, row stride ldc: (C, whether the rest kept its pattern)."""
    M, N, K = A.shape[0], B.shape[0], A.shape[1]
    out_dt = OUT[A.dtype]
    buf = torch.full((M * ldc + 64,), 0x5a5a, dtype=torch.int16, device="cuda")
    Cv = torch.as_strided(buf, (M, N), (ldc, 1), offset).view(out_dt)
    need = abi.mi355_gemm_workspace_bytes(M, N, K, ac.torch_code(A.dtype), ac.AUTO) if workspace else 0
    need += 4 * M * (N + 4) * 16 if workspace and room else 0   # for every plan, also where the query counts on aligned rows
    if ws_bytes is not None:
        need = ws_bytes
    ws = torch.full((max(need, 256),), 0xff, dtype=torch.uint8, device="cuda")
    Ad, Bd = A.cuda(), B.cuda()
    st = abi.mi355_gemm_tn(Ad.data_ptr(), Bd.data_ptr(), Cv.data_ptr(), M, N, K, K, K, ldc, ac.torch_code(A.dtype),
                           ac.torch_code(out_dt), 1.0, ac.AUTO, ws.data_ptr() if need else None, need,
                           torch.cuda.current_stream().cuda_stream)
    assert st == ac.OK
    torch.cuda.synchronize()
    C = Cv.cpu().double()
    Cv.view(torch.int16).fill_(0x5a5a)
    return C, bool((buf == 0x5a5a).all())


def close(C, A, B):
    want = A.double() @ B.double().T
    tol = 3e-2 if A.dtype == torch.float8_e4m3fn else 1e-2
    assert torch.isfinite(C).all()
    assert float((C - want).norm() / want.norm()) <= tol
    # a single wrong or stale element does not hide in the norm: bf16 rounding is 2^-8 of the value, fp32 sums far less
    assert float((C - want).abs().max()) <= 2.0 ** -7 * float(want.abs().max()) + 1e-3


@pytest.mark.parametrize("dt", list(OUT))
@pytest.mark.parametrize("M,N,K", [
    (1, 129, 128), (16, 1001, 512), (17, 4099, 4096),       # streaming kernel, unsplit and split
    (33, 130, 1024), (64, 16897, 2048),                     # its 64-row and its wide tile
    (100, 255, 4096), (128, 4098, 2048),                    # nine-slot ring, K split
    (200, 515, 256), (257, 258, 192),                       # 128 x 128 tiles; a ragged last k-step for fp8
    (512, 8191, 512), (1000, 5037, 768), (1300, 7001, 64),  # several tiles of every shape
])
@pytest.mark.parametrize("offset,pad", [(0, 0), (1, 0), (2, 3), (4, 2)])
def test_ragged_rows(abi, dt, M, N, K, offset, pad):
    A, B = operand(M, K, dt, M + K), operand(N, K, dt, N + K)
    C, kept = run(abi, A, B, offset, N + pad)
    assert kept
    close(C, A, B)


# Small e4m3 products do not get to the kernels that the smaller sizes above are there for; these do.
@pytest.mark.parametrize("M,N,K", [(16, 14333, 592), (30, 14333, 4096), (700, 1303, 192)])   # streaming, unsplit; a ragged last k-step
@pytest.mark.parametrize("offset,pad", [(0, 0), (1, 0), (2, 3), (4, 2)])
def test_ragged_rows_of_large_fp8_products(abi, M, N, K, offset, pad):
    A, B = operand(M, K, torch.float8_e4m3fn, M), operand(N, K, torch.float8_e4m3fn, N)
    C, kept = run(abi, A, B, offset, N + pad)
    assert kept
    close(C, A, B)


def test_aligned_n_in_rows_of_odd_stride_and_address(abi):
    for M, N, K, offset, pad in [(300, 512, 256, 1, 1), (300, 512, 256, 2, 0), (40, 512, 512, 0, 2), (4096, 4096, 128, 1, 0)]:
        A, B = operand(M, K, torch.bfloat16, 1), operand(N, K, torch.bfloat16, 2)
        C, kept = run(abi, A, B, offset, N + pad)
        assert kept
        close(C, A, B)


def close_everywhere(C, A, B):
    """close() with the product in float64 on the GPU, for sizes where the CPU takes long; every element against the bound."""
    want = A.cuda().double() @ B.cuda().double().T
    tol = 3e-2 if A.dtype == torch.float8_e4m3fn else 1e-2
    diff = C.cuda() - want
    assert float(diff.norm() / want.norm()) <= tol
    assert float(diff.abs().max()) <= 2.0 ** -7 * float(want.abs().max()) + 1e-3


# N % 4 == 2; the plan is that of N rounded up to 4: a tail split, or two launches with the second one a few columns or rows.
@pytest.mark.parametrize("M,N,K,dt,pieces", [
    (5000, 3498, 4096, torch.bfloat16, 1), (4352, 4350, 4096, torch.float16, 1), (6144, 4094, 8192, torch.float8_e4m3fn, 1),
    (4096, 4110, 4096, torch.bfloat16, 2), (4110, 4094, 4096, torch.float16, 2), (2304, 8190, 2048, torch.bfloat16, 2),
    (4096, 4110, 8192, torch.float8_e4m3fn, 2)])
def test_tail_split_and_two_pieces(abi, M, N, K, dt, pieces):
    code, Np = ac.torch_code(dt), -(-N // 4) * 4
    cut = [ctypes.c_int64(), ctypes.c_int64()]
    assert abi.mi355_gemm_pieces(M, Np, K, code, ac.AUTO, *[ctypes.byref(x) for x in cut]) == pieces
    assert pieces == 2 or ac.plan(abi, M, Np, K, code)[4] > 0
    A, B = operand(M, K, dt, 3), operand(N, K, dt, 4)
    inner = max(abi.mi355_gemm_workspace_bytes(M, Np, K, code, ac.AUTO), 256)
    # rows at even 2-byte addresses; at odd ones with room for the split's planes only, and with more
    for offset, pad, ws_bytes in ((0, 0, inner), (1, 0, inner), (0, 1, inner), (1, 1, None)):
        C, kept = run(abi, A, B, offset, N + pad, ws_bytes=ws_bytes)
        assert kept
        close_everywhere(C, A, B)


# Rows of C that are aligned, but not by 64 bytes, and a partial last tile column of tiles of 256 rows (4 Mi outputs and more).
@pytest.mark.parametrize("M,N,K,dt", [(908, 10640, 832, torch.float16), (2206, 4076, 1472, torch.bfloat16), (3612, 1516, 4016, torch.float8_e4m3fn),
                                      (5484, 5608, 224, torch.float8_e4m3fn), (2049, 8196, 2048, torch.bfloat16)])
def test_aligned_rows_with_a_partial_last_column(abi, M, N, K, dt):
    A, B = operand(M, K, dt, 27), operand(N, K, dt, 28)
    for offset, pad in ((0, 0), (4, 0), (0, 4), (8, 12)):
        C, kept = run(abi, A, B, offset, N + pad)
        assert kept
        close_everywhere(C, A, B)


# Rows of C at odd 2-byte addresses under plans with tiles of 256 rows: one launch, a tail split, two launches.
@pytest.mark.parametrize("M,N,K,dt", [(2049, 2051, 4096, torch.bfloat16), (513, 8195, 4096, torch.float16), (2049, 6145, 4096, torch.float8_e4m3fn),
                                      (2049, 6145, 2056, torch.bfloat16), (2049, 8195, 4096, torch.bfloat16), (4096, 4111, 4096, torch.bfloat16),
                                      (1025, 6147, 4090, torch.float16)])
def test_rows_at_odd_addresses(abi, M, N, K, dt):
    A, B = operand(M, K, dt, 25), operand(N, K, dt, 26)
    for offset, pad in ((0, 0), (1, 0), (3, 2), (2, 1)):
        C, kept = run(abi, A, B, offset, N + pad)
        assert kept
        close_everywhere(C, A, B)


@pytest.mark.parametrize("workspace", [True, False])
def test_without_a_workspace_too(abi, workspace):
    for M, N, K in [(48, 3001, 1024), (9, 1001, 1024), (100, 203, 2048)]:
        A, B = operand(M, K, torch.bfloat16, 7), operand(N, K, torch.bfloat16, 8)
        C, kept = run(abi, A, B, 0, N, workspace)
        assert kept
        close(C, A, B)


@pytest.mark.parametrize("dt,M,N,K", [(torch.bfloat16, 700, 1030, 513), (torch.float16, 515, 2050, 4100), (torch.float8_e4m3fn, 777, 1001, 1003),
                                      (torch.float8_e4m3fn, 300, 2048, 1025), (torch.float8_e4m3fn, 234, 1568, 1326), (torch.bfloat16, 1024, 1024, 129), (torch.bfloat16, 48, 5001, 4097)])
def test_repacked_operands(abi, dt, M, N, K):
    A, B = operand(M, K, dt, 9), operand(N, K, dt, 10)
    for offset, room in ((0, True), (1, True), (0, False), (1, False)):
        C, kept = run(abi, A, B, offset, N + offset, room=room)
        assert kept
        close(C, A, B)


def test_rows_of_b_farther_apart_than_the_kernels_reach(abi):
    """N % 4 != 0 and 256 rows of B beyond 2 GiB: B is copied to rows that the tiled kernels can address."""
    M, N, K, ldb = 4096, 5, 4096, 1 << 29
    A, B = operand(M, K, torch.bfloat16, 21), operand(N, K, torch.bfloat16, 22)
    far = torch.empty((N - 1) * ldb + K, dtype=torch.bfloat16, device="cuda")
    for n in range(N):
        far[n * ldb:n * ldb + K] = B[n].cuda()
    Ad, C = A.cuda(), torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    need = abi.mi355_gemm_workspace_bytes(M, N, K, ac.BF16, ac.AUTO)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    st = abi.mi355_gemm_tn(Ad.data_ptr(), far.data_ptr(), C.data_ptr(), M, N, K, K, ldb, N, ac.BF16, ac.BF16, 1.0, ac.AUTO,
                           ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    assert st == ac.OK
    close(C.cpu().double(), A, B)


@pytest.mark.parametrize("M,N,K,dt", [(300, 1003, 1024, torch.bfloat16), (65, 514, 2055, torch.float16), (300, 130, 4096, torch.float8_e4m3fn),
                                      (40, 2049, 2048, torch.bfloat16), (260, 1000, 264, torch.bfloat16)])
def test_rows_of_c_farther_apart_than_the_kernels_reach(abi, M, N, K, dt):
    """Computed into a padded copy of C and copied out, on the streaming kernel, the tile kernel and its K splits."""
    A, B = operand(M, K, dt, 23), operand(N, K, dt, 24)
    C, kept = run(abi, A, B, 1, (1 << 21) + 3)
    assert kept
    close(C, A, B)
