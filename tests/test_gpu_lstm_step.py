"""The one-launch time step of LSTM layers whose width is no multiple of 32: edges of its 32 x 8 and 16 x 16 tiles, wavefronts with
no run of k, one or several, and the first size that is too large for it, against the CPU oracle and against the two-launch
path.  Tolerance: rel 1e-4 / abs 1e-5, as for the other LSTM paths."""
import numpy as np
import pytest

from myea_amd import binding as mb
from tests.common import assert_close, run_step
from tests.test_gpu_lstm import ABS, REL, _compare, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,B,Bmax", [(1, 1, 1), (7, 33, 33), (8, 32, 40), (17, 16, 16), (31, 17, 17), (65, 65, 65), (200, 60, 60), (257, 31, 31), (130, 495, 495)])
def test_step_of_any_width(cells, B, Bmax, monkeypatch):
    T = 3
    specs = [dict(units=5), dict(type="lstm", units=cells), dict(units=cells + 2, activation="LINEAR")]
    hyper = dict(type_optimizer_function=mb.OPTIMIZER["AMSGRAD"])
    desc, gpu, cpu = _pair(specs, Bmax, T, hyper, seed=cells, threads=8)
    _, two, _ = _pair(specs, Bmax, T, hyper, seed=cells, threads=8)
    rng = np.random.default_rng(B)
    X, Y = (rng.normal(0, 1, (B, T * w)).astype(np.float32) for w in (5, cells + 2))
    for n in (gpu, cpu):
        run_step(n, B, X, Y, update=False)
    _compare(desc, gpu, cpu, B, T, what="step")
    g, want = gpu.download_gradient(), cpu.download_gradient()
    assert_close(g, want, REL, ABS * max(1.0, float(np.abs(want).max())), what="gradient")
    monkeypatch.setenv("MYEA_LSTM_FUSED", "0")
    run_step(two, B, X, Y, update=False)
    assert_close(g, two.download_gradient(), REL, ABS * max(1.0, float(np.abs(want).max())), what="gradient, one launch against two")


def test_infinite_weight_saturates_a_gate_as_in_fp32():
    """One weight of infinity at a time, recurrent ones and peepholes among them: a gate's sum is an infinity (not NaN) wherever
    what the weight meets is not zero, and the activations of an infinity are finite."""
    T, B, cells = 2, 5, 9
    desc, gpu, _ = _pair([dict(units=4), dict(type="lstm", units=cells), dict(units=cells, activation="LINEAR")], B, T, {}, seed=3)
    w = gpu.download_parameters()
    X = np.random.default_rng(1).normal(0, 1, (B, T * 4)).astype(np.float32)
    layer = desc.layers[1]
    assert layer.last_connection_index - layer.first_connection_index == cells * (4 * (4 + cells) + 3)
    for i in range(layer.first_connection_index, layer.last_connection_index):
        v = w.copy()
        v[i] = np.inf
        gpu.upload_parameters(v)
        gpu.Forward_Pass(B, X)
        assert np.isfinite(gpu.download_tensor(1, mb.TENSOR["OUTPUTS"], T * B * cells)).all(), i
