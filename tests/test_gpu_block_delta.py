"""A residual layer's errors and the delta of its block's last member out of one launch: blocks above each other that keep their width, grow
and shrink, by an even and an odd number of units, in fours and not, with and without a normalisation of the block, time steps and
a batch that leaves rows empty, against the CPU oracle (rel 1e-4 / abs 1e-5
of the largest gradient); the delta is the layer's errors, cropped, bit for bit."""
import numpy as np
import pytest

from myea_amd import binding as mb
from tests.common import assert_close, run_step
from tests.test_gpu_lstm import _pair

pytestmark = pytest.mark.gpu

WIDTHS = [(8, 8, 8), (16, 8, 24), (24, 8, 8), (9, 6, 11), (5, 5, 5), (16, 10, 6), (260, 256, 256)]


@pytest.mark.parametrize("T,B,Bmax", [(1, 7, 7), (3, 4, 4), (3, 3, 5)])
@pytest.mark.parametrize("block_norm", [False, True])
@pytest.mark.parametrize("widths", WIDTHS)
def test_blocks_against_the_oracle(widths, block_norm, T, B, Bmax):
    bn = dict(normalization="BATCH_NORMALIZATION")
    specs = [dict(units=5), dict(units=widths[0], activation="TANH")]
    ends = []
    for w in widths:
        specs += [dict(type="residual", block_depth=2, **(bn if block_norm else {})), dict(units=w, activation="TANH", **bn), dict(units=w, activation="TANH", **bn)]
        ends.append(len(specs) - 1)
    specs += [dict(units=3, activation="LINEAR")]
    desc, gpu, cpu = _pair(specs, Bmax, T, dict(normalization_epsilon=0.1), seed=sum(widths), threads=8)
    rng = np.random.default_rng(B)
    X, Y = (rng.normal(0, 1, (B, T, n)).astype(np.float32) for n in (5, 3))
    for n in (gpu, cpu):
        for _ in range(2):
            run_step(n, B, X, Y, update=False)
    want = cpu.download_gradient()
    assert_close(gpu.download_gradient(), want, 1e-4, 1e-5 * max(1.0, float(np.abs(want).max())), what="gradient")
    if not block_norm:   # the cropped errors themselves
        H = widths[0]
        for end, w in zip(ends, widths):
            H, crop = max(H, w), (H - w + 1) // 2 if H > w else 0
            errors = gpu.download_tensor(end - 2, mb.TENSOR["ERRORS"], T * Bmax * H).reshape(T, Bmax, H)[:, :B]
            delta = gpu.download_tensor(end, mb.TENSOR["ERRORS"], T * Bmax * w).reshape(T, Bmax, w)[:, :B]
            assert np.any(delta) and np.array_equal(delta, errors[:, :, crop:crop + w]), "delta of layer %d" % end
