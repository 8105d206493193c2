"""The short product (few tiles, its wavefronts share k) around the forms its operands are loaded in: whole lines turned round in LDS
against rows straight into the lanes (up to 8 rows of A, or 34 of A and B in a tile), k's that end inside a 16-byte chunk, a run or a round of runs, rows and columns
that end inside a tile, rows that are not 16-byte aligned, four and eight wavefronts - against float64."""
import pytest
import torch

from myea_amd import binding as mb
from tests.test_gpu_gemm_split import LAYOUTS, _operands
from tests.test_gpu_kernels import _gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("M,N", [(1, 77), (8, 256), (9, 33), (14, 20), (15, 20), (70, 2), (70, 3), (40, 95), (333, 500)])
@pytest.mark.parametrize("K", [16, 29, 32, 35, 255, 256, 258, 511, 545, 783])
def test_edges_against_float64(a_kc, b_kc, M, N, K):
    """an accumulator takes one rounding (2^-23 of what it holds, at most the sum of the magnitudes) per 16 k's, a few more join the parts"""
    A, B, Ad, Bd = _operands(a_kc, b_kc, M, N, K, M + N + K)
    # behind the operands' last element: what a load beyond it would bring
    Ad, Bd = (torch.cat([t.flatten(), torch.full((64,), float("nan"), device="cuda")])[:t.numel()].view_as(t) for t in (Ad, Bd))
    C = torch.full((M, N), float("nan"), device="cuda")
    _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, Ad, Bd, C)
    bound = 2.0 ** -23 * (-(-K // 16) + 8) * (A.double().abs() @ B.double().abs())
    assert bool(((C.double() - A.double() @ B.double()).abs() <= bound).all())
