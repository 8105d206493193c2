"""The FP32 contraction on the BF16 matrix cores (three BF16 numbers an operand): every tile shape at its edges and remainders of
a K step against float64, and operands that the split cannot carry (infinities, NaN, values that round to a BF16 infinity)
against what FP32 arithmetic gives."""
import numpy as np
import pytest
import torch

from myea_amd import binding as mb
from tests.test_gpu_kernels import _gemm

pytestmark = pytest.mark.gpu

LAYOUTS = [(1, 1), (1, 0), (0, 0), (0, 1)]
# the tiled kernel, a shape per tile: at least 128 tiles of 64 x 64 (below it is the short product's) and
TILE_64 = [(700, 1000), (1001, 777), (1025, 1030)]   # fewer than 128 of 128 x 128
TILE_64_128, TILE_128_64 = [(1500, 1501), (1409, 1500)], [(3001, 700), (1600, 1500)]   # up to 255 of them
TILE_128 = [(2049, 2050), (2180, 1921)]
# k's at, around and beyond a step of 16 or 32, and for the 64 x 64 tile around the four steps that it keeps in registers
SHAPES = ([t + (k,) for t in TILE_64 for k in (16, 31, 33, 65, 127, 161, 257, 545)] + [t + (k,) for t in TILE_64_128 + TILE_128_64 for k in (16, 31, 65, 97)] +
          [t + (k,) for t in TILE_128 for k in (17, 48, 95)] + [(33100, 33, 65), (50, 33000, 33)] +   # thin: 128 x 64 and 64 x 128
          [(190, 1100, 1), (65, 1300, 15), (600, 640, 33)])   # shallow, shallow, short


def _operands(a_kc, b_kc, M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A, B = torch.randn((M, K), generator=g, device="cuda"), torch.randn((K, N), generator=g, device="cuda")
    return A, B, (A if a_kc else A.t()).contiguous(), (B.t() if b_kc else B).contiguous()


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tiles_and_remainders_against_float64(a_kc, b_kc, M, N, K):
    """An accumulator takes one rounding (2^-23 of what it holds, at most the sum of the magnitudes) per 16 k's, a few more join
    the parts; the products left out are below 2^-24 of theirs."""
    A, B, Ad, Bd = _operands(a_kc, b_kc, M, N, K, M + N + K)
    C = torch.full((M, N), float("nan"), device="cuda")
    _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, Ad, Bd, C)
    bound = 2.0 ** -23 * (-(-K // 16) + 8) * (A.double().abs() @ B.double().abs())
    assert bool(((C.double() - A.double() @ B.double()).abs() <= bound).all())


@pytest.mark.parametrize("M,N", [(96, 100), (640, 768), (1030, 1000), (2049, 2050)])   # short (eight and four wavefronts), 64 x 64, 128 x 128
def test_error_over_many_products(M, N):
    """2-norm of the error over that of the result at k = 4096: what myea_gemm.hip states for the tiled kernel is 4.0e-7 for normal operands
    (two planes of BF16 would leave 3.5e-6, emulated) and 3.1e-7 for positive ones (a unit that cut its sums off where this one rounds them
    would leave 5.7e-6, emulated); the FP32 instruction has 1.15e-6 and 8.4e-7.  The short product adds
    four or eight shorter sums and is below both."""
    K = 4096
    A, B, _, _ = _operands(1, 1, M, N, K, M)
    for a, b, most in ((A, B, 5e-7), (A.abs(), B.abs(), 4e-7)):
        C = torch.empty((M, N), device="cuda")
        _gemm(mb.load_library(), 1, 1, 0, M, N, K, a, b.t().contiguous(), C)
        want = a.double() @ b.double()
        assert ((C.double() - want).norm() / want.norm()).item() <= most


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(100, 90, 300), (1000, 700, 97), (1500, 1501, 40), (2049, 2050, 40)])
def test_small_operands_keep_their_bits(a_kc, b_kc, M, N, K):
    """One operand down to FP32's subnormals, the other large or ordinary: the products are as exact as any, but for results that
    are subnormal themselves (one rounding more, 2^-149)."""
    A, B, _, _ = _operands(a_kc, b_kc, M, N, K, 11)
    for at_a, at_b in ((-115, 100), (90, -126), (-140, 100), (-120, 0), (0, -146)):
        a, b = (A.double() * 2.0 ** at_a).float(), (B.double() * 2.0 ** at_b).float()
        C = torch.full((M, N), float("nan"), device="cuda")
        _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, (a if a_kc else a.t()).contiguous(), (b.t() if b_kc else b).contiguous(), C)
        bound = 2.0 ** -23 * (-(-K // 16) + 8) * (a.double().abs() @ b.double().abs()) + 2.0 ** -149
        inside = bool(((C.double() - a.double() @ b.double()).abs() <= bound).all())
        assert inside, (at_a, at_b)


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 11, 15])
def test_shallow_products_are_rounded_once(a_kc, b_kc, K):
    """Fewer k's than a BF16 instruction's 16: the sum is held in 64 bits, so a result is its FP32 neighbour (half an ulp, and 2^-50 of
    the magnitudes for the 64-bit sums on both sides) - over heavy-tailed, subnormal, overflowing and infinite values, onto C as well."""
    for M, N in ((1, 1), (31, 33), (32, 32), (65, 100), (300, 33), (100, 4097), (1025, 700)):
        A, B, _, _ = _operands(a_kc, b_kc, M, N, K, M + N + K)
        A, B = A * torch.exp(4 * A), B.clone()
        A[0, 0], B[K - 1, N // 2] = 1e-42, -3e38
        Ad, Bd = (A if a_kc else A.t()).contiguous(), (B.t() if b_kc else B).contiguous()
        C = torch.full((M, N), float("nan"), device="cuda")
        _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, Ad, Bd, C)
        want, magnitude = A.double() @ B.double(), A.double().abs() @ B.double().abs()
        finite = want.abs() < 3.4e38
        off = (C.double() - want).abs() > 2.0 ** -24 * want.abs() + 2.0 ** -50 * magnitude + 2.0 ** -150
        assert not bool((off & finite).any()) and bool((C[want.abs() > 3.5e38].isinf()).all()), (M, N)
        D = torch.ones((M, N), device="cuda")
        _gemm(mb.load_library(), a_kc, b_kc, 1, M, N, K, Ad, Bd, D)
        assert torch.equal(D, C + 1), (M, N)
        A[M // 2, 0], B[0, 0] = float("inf"), float("nan")
        _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, (A if a_kc else A.t()).contiguous(), (B.t() if b_kc else B).contiguous(), C)
        want = (A.double() @ B.double()).float()
        assert torch.equal(C.isnan(), want.isnan()) and torch.equal(C.isinf() & (C > 0), want.isinf() & (want > 0)), (M, N)


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("M,N", [(100, 90), (700, 1000), (1500, 1501), (1600, 1500), (2049, 2050)])
def test_values_the_split_cannot_carry(a_kc, b_kc, M, N):
    K = 40
    A, B, _, _ = _operands(a_kc, b_kc, M, N, K, 3)
    A[3, 5], A[10, 39], B[0, 20], A[50, 0], A[60] = float("inf"), float("nan"), -float("inf"), 3.4e38, 0.0
    B[0, :20] = 0.25   # 3.4e38 rounds to a BF16 infinity; its products here are finite
    Ad, Bd = (A if a_kc else A.t()).contiguous(), (B.t() if b_kc else B).contiguous()
    C = torch.zeros((M, N), device="cuda")
    _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, Ad, Bd, C)
    want, got = (A.cpu().double() @ B.cpu().double()).float().numpy(), C.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    infinite = np.isinf(want)
    assert np.array_equal(np.isinf(got), infinite) and np.array_equal(got[infinite], want[infinite])
    finite = np.isfinite(want)
    magnitudes = (np.nan_to_num(A.abs().cpu().double().numpy(), posinf=0.0)) @ (np.nan_to_num(B.abs().cpu().double().numpy(), posinf=0.0))
    assert np.all(np.abs(got[finite].astype(np.float64) - want[finite]) <= 2.0 ** -23 * (K + 8) * magnitudes[finite])


@pytest.mark.parametrize("a_kc,b_kc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(1, 33, 1), (31, 1, 23), (33, 32, 24), (32, 65, 31), (64, 64, 33), (95, 100, 255), (100, 31, 257), (500, 490, 545),
                                   (257, 1000, 17), (700, 600, 33), (700, 600, 545), (512, 1024, 129), (30, 16300, 300), (520, 1000, 300)])
def test_short_products_against_float64(a_kc, b_kc, M, N, K):
    """Fewer than 128 tiles of 64 x 64: workgroups of 32 x 32, of eight wavefronts up to 256 of them and of four beyond, that share k in runs
    of 32, of which the last ones may have none or a part; the last three shapes are the tiled kernel's."""
    A, B, Ad, Bd = _operands(a_kc, b_kc, M, N, K, M + N + K)
    C = torch.full((M, N), float("nan"), device="cuda")
    _gemm(mb.load_library(), a_kc, b_kc, 0, M, N, K, Ad, Bd, C)
    bound = 2.0 ** -23 * (-(-K // 16) + 8) * (A.double().abs() @ B.double().abs())
    assert bool(((C.double() - A.double() @ B.double()).abs() <= bound).all())


def test_pair_of_odd_widths_matches_the_separate_launches():
    """Rows that are no 16-byte multiples ride in the paired launch too: 128 tiles of dX beside 256 of dW, bit for bit."""
    from tests.test_gpu_paired_backward import _pair, _step
    B = 1021
    specs = [dict(units=2045), dict(units=2047, activation="RELU"), dict(units=2047, activation="TANH"), dict(units=5, activation="LINEAR")]
    desc, (a, b), X, Y, _ = _pair(specs, B)
    b.profile_enable(True)
    for _ in range(2):
        _step(a, B, X, Y, fused=False)
        _step(b, B, X, Y, fused=True)
    pairs = b.profile_read(4)
    b.profile_enable(False)
    assert pairs[0] >= 2, pairs
    assert np.array_equal(a.download_gradient(), b.download_gradient())
    for li in range(1, desc.n_layers):
        assert np.array_equal(a.download_tensor(li, mb.TENSOR["ERRORS"]), b.download_tensor(li, mb.TENSOR["ERRORS"]))
