"""A single time step's normalisation of a residual block's members as one launch, forward (with the activation and the dropout multiplier
in it) and backward (the scale's and the shift's gradient straight onto the gradient, and added to on a second pass), at the edges of its
column groups and of the sizes it is taken for, against the CPU oracle: rel 1e-4 / abs 1e-5."""
import numpy as np
import pytest

from myea_amd import binding as mb
from tests.common import assert_close, run_step
from tests.test_gpu_lstm import _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norm", ["BATCH_NORMALIZATION", "BATCH_RENORMALIZATION"])
@pytest.mark.parametrize("units,B,Bmax", [(3, 5, 5), (4, 64, 70), (7, 65, 65), (130, 512, 512), (33, 513, 513), (1025, 24, 24)])
def test_members_against_the_oracle(norm, units, B, Bmax):
    bn = dict(normalization=norm)
    block = [dict(type="residual", block_depth=2), dict(units=units, activation="TANH", **bn), dict(units=units, activation="TANH", dropout="BERNOULLI_INVERTED", keep=0.5, **bn)]
    specs = [dict(units=9), dict(units=units, activation="TANH")] + block + [dict(units=4, activation="SOFTMAX")]
    desc, gpu, cpu = _pair(specs, Bmax, 1, dict(type_loss_function=mb.LOSS["CROSS_ENTROPY"], normalization_epsilon=0.1), seed=units, threads=8)
    rng = np.random.default_rng(B)
    masks = (rng.random(desc.total_mask_units) < 0.6).astype(np.uint8)
    X = rng.normal(0, 1, (B, 9)).astype(np.float32)
    Y = np.eye(4, dtype=np.float32)[rng.integers(0, 4, B)]
    for n in (gpu, cpu):
        n.upload_masks(masks)
        for _ in range(2):   # the second adds to the first
            run_step(n, B, X, Y, update=False)
    for li in range(3, 5):
        W = units
        a, b = (n.download_tensor(li, mb.TENSOR["OUTPUTS"], Bmax * W).reshape(Bmax, W)[:B] for n in (gpu, cpu))
        assert_close(a, b, 1e-4, 1e-5, what="outputs of layer %d" % li)
    want = cpu.download_gradient()
    assert_close(gpu.download_gradient(), want, 1e-4, 1e-5 * max(1.0, float(np.abs(want).max())), what="gradient")
