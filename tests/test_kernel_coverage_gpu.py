"""The cases of kernel_coverage_cases.py, element by element: sums of small integers are exact."""
import pytest
import torch

from tests import abi_ctypes as ac, test_cut_gpu
from tests.kernel_coverage_cases import MX, ODD_ROWS, REPACKED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", MX)
def test_mx(M, N, K):
    test_cut_gpu.test_block_scaled(M, N, K)


@pytest.mark.parametrize("M,N,K,dt", ODD_ROWS + REPACKED)
def test_rows_of_any_alignment(M, N, K, dt):
    test_cut_gpu.test_plain(M, N, K, {ac.BF16: torch.bfloat16, ac.E4M3: torch.float8_e4m3fn}[dt])
