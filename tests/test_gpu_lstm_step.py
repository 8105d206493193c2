"""The one-launch time step of LSTM layers whose width is no multiple of 32: edges of its 32 x 8 and 16 x 16 tiles, wavefronts with
no run of k, one or several, and the first size that is too large for it, against the CPU oracle and against the two-launch
path.  Tolerance: rel 1e-4 / abs 1e-5, as for the other LSTM paths."""
import numpy as np
import pytest

from myea_amd import binding as mb
from tests.common import assert_close, glorot_parameters, run_step
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


def test_infinite_weight_saturates_a_gate_as_in_fp32(monkeypatch):
    """One weight of infinity at a time, recurrent ones and peepholes among them: a gate's sum is an infinity (not NaN) wherever
    what the weight meets is not zero, and the activations of an infinity are finite - the same as through the two launches."""
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
        out = []
        for fused in ("1", "0"):
            monkeypatch.setenv("MYEA_LSTM_FUSED", fused)
            gpu.Forward_Pass(B, X)
            out.append(gpu.download_tensor(1, mb.TENSOR["OUTPUTS"], T * B * cells))
        assert np.isfinite(out[0]).all(), i
        assert_close(out[0], out[1], REL, ABS, what="weight %d" % i)


@pytest.mark.parametrize("cells,B", [(9, 5), (130, 40)])
def test_recurrent_weights_below_the_split_range_keep_their_bits(cells, B):
    """Recurrent weights of 2^-120 between ordinary gate deltas: with no error from above at the first of two steps, dh there is
    dG[1] Wrec alone, held against 64 bits (4 cells products: 2^-23 of their magnitudes per rounding, one per 32 k's and the sum of
    the 16 wavefronts)."""
    T, In = 2, 4
    desc = mb.make_desc([dict(units=In), dict(type="lstm", units=cells), dict(units=cells, activation="LINEAR")], B, T)
    net = mb.HipNetwork(desc, mb.default_hyper(type_loss_function=mb.LOSS["MSE"]))
    net.set_state_propagation(mb.STATE_TRAINING)
    w = glorot_parameters(desc, 4, bias_range=0.3)
    layer, rows = desc.layers[1], In + cells
    per_cell = w[layer.first_connection_index:layer.last_connection_index].reshape(cells, 4 * rows + 3)
    # a cell's slice: its input row [In + cells], the three gates' rows from below, then their recurrent rows, the peepholes
    recurrent = [per_cell[:, In:rows]] + [per_cell[:, rows + 3 * In + g * cells:rows + 3 * In + (g + 1) * cells] for g in range(3)]
    for r in recurrent:
        r *= np.float32(2.0 ** -120)
    net.upload_parameters(w)
    net.Clear_Training_Arrays()
    X = np.random.default_rng(1).normal(0, 1, (B, T * In)).astype(np.float32)
    net.Forward_Pass(B, X)
    Y = net.download_tensor(2, mb.TENSOR["OUTPUTS"]).reshape(T, B, cells).copy()
    Y[1] += np.random.default_rng(2).normal(0, 1, (B, cells)).astype(np.float32)
    net.Compute__Error(B, np.ascontiguousarray(Y.transpose(1, 0, 2)).reshape(B, T * cells))
    net.Backward_Pass(B)
    taps = ["LSTM_DELTA_CELL_INPUT", "LSTM_DELTA_INPUT_GATE", "LSTM_DELTA_FORGET_GATE", "LSTM_DELTA_OUTPUT_GATE"]
    dG = [net.download_tensor(1, mb.TENSOR[t], T * B * cells).reshape(T, B, cells)[1].astype(np.float64) for t in taps]
    got = net.download_tensor(1, mb.TENSOR["ERRORS"]).reshape(T, B, cells)[0].astype(np.float64)
    want = sum(d @ r.astype(np.float64) for d, r in zip(dG, recurrent))
    magnitude = sum(np.abs(d) @ np.abs(r.astype(np.float64)) for d, r in zip(dG, recurrent))
    assert np.abs(want).max() > 0
    assert np.all(np.abs(got - want) <= 2.0 ** -23 * (cells / 8 + 20) * magnitude + 2.0 ** -149)
