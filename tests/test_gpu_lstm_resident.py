"""The LSTM time loop as one resident launch per layer and pass, through the C ABI: against the same library with one launch per time step
(MYEA_LSTM_RESIDENT=0), against the CPU oracle, and the bounded wait's give-up path.  Up to 512 cells the loops run on the BF16 matrix
cores; the FP32 instruction has the backward loop of 512 cells at more than one row of 16 examples a group, in two forms - a member's two chains
in two sets of wavefronts, or (MYEA_LSTM_BACKWARD_SETS=0) in one instruction stream - and both loops of 1024.
Tolerance rel 1e-4 / abs 1e-5 (the resident kernels use the exp2 and reciprocal instructions in the gate functions, the
per-step kernels expf and a division: a few ulp apart)."""
import ctypes as C

import numpy as np
import pytest

from myea_amd import binding as mb
from tests.common import assert_close, environment, glorot_parameters, run_step
from tests.oracle_lib import OracleNetwork
from tests.test_gpu_lstm import LSTM_TAPS, _rows, _width

pytestmark = pytest.mark.gpu
REL, ABS = 1e-4, 1e-5
BACK = mb.TENSOR["DIRECTION_BACKWARD"]
FORWARD_LOOP, BACKWARD_LOOP = 5, 6   # profile families of the time loops


lstm = lambda units, **kw: dict(type="lstm", units=units, **kw)
zone = lambda units, **kw: dict(type="lstm", units=units, dropout="ZONEOUT", keep=0.3, keep_output=0.2, **kw)

class PlanesPlan(C.Structure):
    _fields_ = [("ok", C.c_bool), ("backward", C.c_bool)] + [(n, C.c_int) for n in ("members", "rs", "row_tiles", "row_groups", "grid", "cus")]


def planes_plan(cells, B, dirs=1):
    """how a layer runs on the BF16 matrix cores: ok (forward) and backward say whether it does, rs how many row tiles a group has"""
    plan_of = getattr(mb.load_library(), "_ZN4myea16lstm_planes_planEmmmmiPNS_14LstmPlanesPlanE")
    plan_of.argtypes = [C.c_size_t] * 4 + [C.c_int, C.POINTER(PlanesPlan)]
    plan = PlanesPlan()
    assert plan_of(cells, 1, B, B, dirs, C.byref(plan)) == 0
    return plan


def _fp32_backward(layers, B):
    """the FP32 instruction has the backward loop of the layers that have a loop of 512 or 1024 cells"""
    return [not planes_plan(_width(l), B, 2 if l.use_bidirectional else 1).backward for l in layers]


# name, layers, T, B, Bmax, which layers' backward loops are the FP32 instruction's
CASES = [
    ("128-cells-last-chain-ragged", [dict(units=24), lstm(128), dict(units=128, activation="LINEAR")], 9, 70, 72, [False]),
    ("128-cells-second-chain-empty", [dict(units=8), lstm(128), dict(units=128, activation="LINEAR")], 5, 13, 16, [False]),
    ("256-cells-two-directions", [dict(units=12), lstm(256, bidirectional=True), dict(units=256, activation="TANH")], 5, 33, 40, [False]),
    ("512-cells-zoneout-stacked", [dict(units=16), zone(512), lstm(128), dict(units=128, activation="LINEAR")], 4, 48, 48, [False, False]),
    ("512-cells-two-directions-ragged", [dict(units=9), lstm(512, bidirectional=True), dict(units=512, activation="LINEAR")], 4, 41, 44, [False]),
    ("512-cells-beyond-a-row-zoneout-stacked", [dict(units=16), zone(512), lstm(128), dict(units=128, activation="LINEAR")], 4, 141, 144, [True, False]),
    ("512-cells-beyond-a-row-two-directions", [dict(units=9), lstm(512, bidirectional=True), dict(units=512, activation="LINEAR")], 4, 70, 70, [True]),
    ("512-cells-beyond-a-row-two-directions-zoneout", [dict(units=7), zone(512, bidirectional=True), dict(units=512, activation="LINEAR")], 6, 128, 128, [True]),
    ("512-cells-beyond-a-row-two-steps", [dict(units=5), lstm(512), dict(units=512, activation="LINEAR")], 2, 256, 256, [True]),
    ("1024-cells-two-directions", [dict(units=10), lstm(1024, bidirectional=True), dict(units=1024, activation="LINEAR")], 3, 40, 40, [True]),
    ("1024-cells-ragged-seven-steps", [dict(units=6), lstm(1024), dict(units=1024, activation="LINEAR")], 7, 45, 48, [True]),
    ("1024-cells-two-steps", [dict(units=5), lstm(1024), dict(units=1024, activation="LINEAR")], 2, 33, 33, [True]),
    ("1024-cells-twelve-steps-zoneout", [dict(units=7), zone(1024, bidirectional=True), dict(units=1024, activation="LINEAR")], 12, 64, 64, [True]),
    ("two-steps", [dict(units=6), lstm(256), dict(units=256, activation="LINEAR")], 2, 32, 32, [False]),
]


def _net(desc, h, w, masks):
    n = mb.HipNetwork(desc, h)
    n.set_state_propagation(mb.STATE_TRAINING)
    n.upload_parameters(w)
    if masks is not None:
        n.upload_zoneout_masks(masks)
    n.Clear_Training_Arrays()
    return n


def _setup(specs, T, B, Bmax, seed):
    desc = mb.make_desc(specs, Bmax, T)
    h = mb.default_hyper(type_optimizer_function=mb.OPTIMIZER["ADAM"], type_loss_function=mb.LOSS["MSE"])
    w = glorot_parameters(desc, seed, bias_range=0.3)
    rng = np.random.default_rng(seed)
    masks = None
    if any(s.get("dropout") == "ZONEOUT" for s in specs):
        cells = sum(_width(desc.layers[i]) * (2 if desc.layers[i].use_bidirectional else 1)
                    for i in range(desc.n_layers) if desc.layers[i].type_layer == mb.LAYER_LSTM)
        masks = (rng.uniform(0, 1, 2 * T * cells) < 0.6).astype(np.uint8)
    X = rng.normal(0, 1, (B, T * specs[0]["units"])).astype(np.float32)
    Y = rng.normal(0, 1, (B, T * specs[-1]["units"])).astype(np.float32)
    return desc, h, w, masks, X, Y


def _compare(desc, a_net, b_net, B, T, what):
    Bmax = desc.batch_size
    for li in range(1, desc.n_layers):
        l = desc.layers[li]
        W = _width(l)
        kinds = [("OUTPUTS", 0), ("ERRORS", 0)]
        if l.type_layer == mb.LAYER_LSTM:
            for flag in ((0, BACK) if l.use_bidirectional else (0,)):
                kinds += [(k, flag) for k in LSTM_TAPS + ["LSTM_CELL_OUTPUT", "LSTM_DELTA_CELL_OUTPUT"]]
        for kind, flag in kinds:
            a = a_net.download_tensor(li, mb.TENSOR[kind] | flag, T * Bmax * W)
            b = b_net.download_tensor(li, mb.TENSOR[kind] | flag, T * Bmax * W)
            assert_close(_rows(a, T, Bmax, B, W), _rows(b, T, Bmax, B, W), REL, ABS, what="%s layer %d %s/%d" % (what, li, kind, flag))
    g = b_net.download_gradient()
    assert_close(a_net.download_gradient(), g, REL, ABS * max(1.0, float(np.abs(g).max())), what=what + " gradient")


def _loop_launches(net):
    return net.profile_read(FORWARD_LOOP)[0], net.profile_read(BACKWARD_LOOP)[0]


LOOP_CASES = [c + ("1",) for c in CASES] + [c + ("0",) for c in CASES if "beyond-a-row" in c[0]]
LOOP_IDS = [c[0] + ("" if c[-1] == "1" else "-one-stream") for c in LOOP_CASES]


@pytest.mark.parametrize("name,specs,T,B,Bmax,fp32,sets", LOOP_CASES, ids=LOOP_IDS)
def test_resident_loop_matches_one_launch_per_step_and_the_oracle(name, specs, T, B, Bmax, fp32, sets):
    desc, h, w, masks, X, Y = _setup(specs, T, B, Bmax, seed=21)
    resident = _net(desc, h, w, masks)
    stepwise = _net(desc, h, w, masks)
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    if masks is not None:
        cpu.upload_zoneout_masks(masks)
    cpu.Clear_Training_Arrays()
    layers = [desc.layers[i] for i in range(desc.n_layers) if desc.layers[i].type_layer == mb.LAYER_LSTM]
    assert _fp32_backward(layers, B) == fp32
    per_step = sum((2 if l.use_bidirectional else 1) * (T - 1) for l in layers)
    for step in range(2):
        with environment(MYEA_LSTM_BACKWARD_SETS=sets):
            resident.profile_enable(True)
            resident.Reset__Loss()
            run_step(resident, B, X, Y, update=False)
            fwd, bwd = _loop_launches(resident)
            resident.profile_enable(False)
        assert fwd == len(layers), "the forward time loops did not run as one launch per layer"
        assert bwd == len(layers), "the backward time loops did not run as one launch per layer"
        with environment(MYEA_LSTM_RESIDENT=0):
            stepwise.profile_enable(True)
            stepwise.Reset__Loss()
            run_step(stepwise, B, X, Y, update=False)
            assert _loop_launches(stepwise) == (per_step, per_step)
            stepwise.profile_enable(False)
        cpu.Reset__Loss()
        run_step(cpu, B, X, Y, update=False)
        _compare(desc, resident, stepwise, B, T, "step %d, resident vs per-step" % step)
        _compare(desc, resident, cpu, B, T, "step %d, resident vs oracle" % step)
        assert resident.get_loss().loss_values == pytest.approx(cpu.get_loss().loss_values, rel=1e-4)
        for n in (resident, stepwise, cpu):
            n.Update_Parameter(B, B)
        wc = cpu.download_parameters()
        resident.upload_parameters(wc)
        stepwise.upload_parameters(wc)


@pytest.mark.parametrize("specs,T,Bmax,batches,fp32,sets", [
    ([dict(units=12), lstm(256, bidirectional=True), lstm(128), dict(units=128, activation="LINEAR")], 7, 80, (80, 45), (False, False), "1"),
    ([dict(units=12), lstm(512, bidirectional=True), dict(units=512, activation="LINEAR")], 5, 128, (128, 70, 41), (True, True, False), "1"),
    ([dict(units=12), lstm(512), dict(units=512, activation="LINEAR")], 5, 150, (150, 129), (True, True), "0"),
    ([dict(units=12), lstm(1024), dict(units=1024, activation="LINEAR")], 3, 60, (60, 20), (True, True), "1"),
], ids=["256-and-128-cells", "512-cells-two-directions", "512-cells-one-stream", "1024-cells"])
def test_bias_and_peephole_gradients_summed_inside_the_backward_loop(specs, T, Bmax, batches, fp32, sets):
    """the resident backward loop sums the bias and peephole gradients of its layer as it goes; MYEA_LSTM_RESIDENT_SUMS=0 has the
    weight-gradient pass read the gate deltas once more instead: the same gradient either way, with examples missing from the last
    group, in both directions, and when a smaller batch follows a larger one"""
    desc, h, w, masks, X, Y = _setup(specs, T, Bmax, Bmax, seed=33)
    inside, apart = _net(desc, h, w, None), _net(desc, h, w, None)
    layers = [desc.layers[i] for i in range(desc.n_layers) if desc.layers[i].type_layer == mb.LAYER_LSTM]
    for B, at in zip(batches, fp32):
        assert _fp32_backward(layers, B) == [at] * len(layers)
        with environment(MYEA_LSTM_BACKWARD_SETS=sets):
            inside.profile_enable(True)
            run_step(inside, B, X[:B], Y[:B], update=False)
            assert _loop_launches(inside)[1] == len(layers), "the backward time loops did not run as one launch per layer"
            inside.profile_enable(False)
            with environment(MYEA_LSTM_RESIDENT_SUMS="0"):
                run_step(apart, B, X[:B], Y[:B], update=False)
        g = apart.download_gradient()
        assert np.abs(g).max() > 0
        assert_close(inside.download_gradient(), g, 2e-5, 2e-6 * float(np.abs(g).max()), what="batch %d: sums inside the loop against the separate pass" % B)
        for n in (inside, apart):
            n.Update_Parameter(B, B)


LATE_CASES = [c for c in CASES if True in c[5]]


@pytest.mark.parametrize("name,specs,T,B,Bmax,fp32", LATE_CASES, ids=[c[0] for c in LATE_CASES])
def test_the_path_of_a_late_group(name, specs, T, B, Bmax, fp32):
    """On the FP32 instruction (1024 cells; the backward loop of 512 in one instruction stream) a unit requests the next unit's first tiles
    between its own last MFMAs if the other chain's counter is complete by then, behind them if not; which of the two happens
    depends on timing.  Here the second is forced (every unit is told "not yet") and held against the oracle."""
    desc, h, w, masks, X, Y = _setup(specs, T, B, Bmax, seed=23)
    zone_masks = masks if any(s.get("dropout") == "ZONEOUT" for s in specs) else None
    gpu = _net(desc, h, w, zone_masks)
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    if zone_masks is not None:
        cpu.upload_zoneout_masks(zone_masks)
    cpu.Clear_Training_Arrays()
    with environment(MYEA_LSTM_RESIDENT_TEST_NEVER_EARLY=1, MYEA_LSTM_BACKWARD_SETS=0):
        gpu.profile_enable(True)
        for n in (gpu, cpu):
            n.Reset__Loss()
            run_step(n, B, X[:B], Y[:B], update=False)
        fwd, bwd = _loop_launches(gpu)
        gpu.profile_enable(False)
    layers = [desc.layers[i] for i in range(desc.n_layers) if desc.layers[i].type_layer == mb.LAYER_LSTM]
    assert fwd == len(layers) and bwd == len(layers), "the time loops did not run as one launch per layer"
    assert _fp32_backward(layers, B) == fp32
    _compare(desc, gpu, cpu, B, T, "late path")


def test_a_smaller_batch_after_a_larger_one():
    """rows beyond the batch keep what the larger batch left there; the rows of the batch do not depend on them"""
    specs = [dict(units=8), lstm(128), dict(units=128, activation="LINEAR")]
    T, Bmax = 6, 64
    desc, h, w, masks, X, Y = _setup(specs, T, Bmax, Bmax, seed=5)
    gpu = _net(desc, h, w, None)
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    cpu.Clear_Training_Arrays()
    for B in (64, 19, 33):
        for n in (gpu, cpu):
            n.Clear_Training_Arrays()
            n.Reset__Loss()
            run_step(n, B, X[:B], Y[:B], update=False)
        _compare(desc, gpu, cpu, B, T, "batch %d" % B)


@pytest.mark.parametrize("cells,B,tiles", [(128, 32, 1), (300, 200, 2), (1024, 32, 0)], ids=["128-cells", "300-cells-two-row-tiles-a-group", "1024-cells-across-two-xcds"])
def test_a_wait_that_gives_up_is_reported_once_and_the_network_carries_on_per_step(cells, B, tiles):
    """Every group is told to expect a member that does not exist: the first wait between time steps runs out of polls,
    every wavefront leaves through the give-up path, the next call that looks reports MYEA_E_DEVICE, and from then on the
    network uses one launch per time step."""
    specs = [dict(units=8), lstm(cells), dict(units=cells, activation="LINEAR")]
    T = 5
    plan = planes_plan(cells, B)
    assert (plan.rs if plan.ok else 0) == tiles
    desc, h, w, masks, X, Y = _setup(specs, T, B, B, seed=7)
    gpu = _net(desc, h, w, None)
    with environment(MYEA_LSTM_RESIDENT_TEST_ABSENT_MEMBER=1, MYEA_LSTM_RESIDENT_SPIN_POLLS=64):
        gpu.Forward_Pass(B, X)
        with pytest.raises(mb.MyeaError) as e:
            gpu.synchronize()
    assert e.value.code == mb.E_DEVICE and "gave up" in str(e.value)
    gpu.synchronize()   # reported once
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    cpu.Clear_Training_Arrays()
    gpu.profile_enable(True)
    for n in (gpu, cpu):
        n.Clear_Training_Arrays()
        n.Reset__Loss()
        run_step(n, B, X, Y, update=False)
    assert _loop_launches(gpu) == (T - 1, T - 1), "after a give-up the time loops run one launch per step"
    gpu.profile_enable(False)
    _compare(desc, gpu, cpu, B, T, "after the give-up")


# the row tiles a group has on the BF16 matrix cores, 0: the FP32 instruction's loop
@pytest.mark.parametrize("cells,B,tiles,sets", [(128, 32, 1, "1"), (300, 200, 2, "1"), (512, 32, 1, "1"), (512, 141, 0, "1"), (512, 141, 0, "0"), (1024, 32, 0, "1")],
                         ids=["128-cells", "300-cells-two-row-tiles-a-group", "512-cells", "512-cells-a-set-of-wavefronts-per-chain", "512-cells-one-stream",
                              "1024-cells-across-two-xcds"])
def test_a_backward_wait_that_gives_up_is_reported_too(cells, B, tiles, sets):
    """the same forced give-up in the backward loop, in each of its forms (on the FP32 instruction with tile loads into LDS in flight when the
    wait begins; in the form of two sets of wavefronts every wait - for the group, for the turn, for each other - runs out on its own):
    the forward pass runs normally, the backward loop's first wait between steps runs out of polls and every wavefront leaves"""
    specs = [dict(units=8), lstm(cells), dict(units=cells, activation="LINEAR")]
    T = 5
    plan = planes_plan(cells, B)
    assert (plan.rs if plan.backward else 0) == tiles
    desc, h, w, masks, X, Y = _setup(specs, T, B, B, seed=9)
    gpu = _net(desc, h, w, None)
    gpu.Forward_Pass(B, X)
    gpu.Compute__Error(B, Y)
    gpu.synchronize()
    with environment(MYEA_LSTM_RESIDENT_TEST_ABSENT_MEMBER=1, MYEA_LSTM_RESIDENT_SPIN_POLLS=64, MYEA_LSTM_BACKWARD_SETS=sets):
        gpu.Backward_Pass(B)
        with pytest.raises(mb.MyeaError) as e:
            gpu.synchronize()
    assert e.value.code == mb.E_DEVICE and "gave up" in str(e.value)
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    cpu.Clear_Training_Arrays()
    for n in (gpu, cpu):
        n.Clear_Training_Arrays()
        n.Reset__Loss()
        run_step(n, B, X, Y, update=False)
    _compare(desc, gpu, cpu, B, T, "after the backward give-up")


# a layer's backward loop leaves half of the 256 compute units: groups of 16 examples on the BF16 matrix cores (one to an XCD until they
# are more than eight), of 32 at 1024 cells (64 workgroups each)
@pytest.mark.parametrize("cells,B,dirs,room", [(1024, 1, 1, True), (1024, 64, 1, True), (1024, 65, 1, False), (256, 128, 1, True), (256, 129, 1, False),
                                               (200, 60, 1, True), (512, 16, 1, False), (512, 141, 1, False), (1000, 16, 1, False)])
def test_which_loops_leave_room_for_contractions_beside_them(cells, B, dirs, room):
    leaves_room = getattr(mb.load_library(), "_ZN4myea25lstm_backward_leaves_roomEmmmmi")
    leaves_room.argtypes, leaves_room.restype = [C.c_size_t] * 4 + [C.c_int], C.c_bool
    assert leaves_room(cells, 1, B, B, dirs) == room


@pytest.mark.parametrize("cells", [128, 1024])
def test_weight_contractions_beside_the_backward_loop_change_nothing(cells):
    """the combined backward + weight-gradient call runs the weight contractions of the layer above on a second stream beside an
    LSTM layer's backward time loop: same gradient as the two separate calls, and the same as the oracle"""
    specs = [dict(units=16), lstm(cells), lstm(cells), dict(units=cells, activation="LINEAR")]
    T, B = 6, 64
    desc, h, w, masks, X, Y = _setup(specs, T, B, B, seed=13)
    combined, separate = _net(desc, h, w, None), _net(desc, h, w, None)
    cpu = OracleNetwork(desc, h, threads=8)
    cpu.set_state_propagation(mb.STATE_TRAINING)
    cpu.upload_parameters(w)
    cpu.Clear_Training_Arrays()
    for step in range(2):
        combined.Forward_Pass(B, X)
        combined.Compute__Error(B, Y)
        combined.Backward_Pass__Update_Derivative_Weight(B)
        run_step(separate, B, X, Y, update=False)
        run_step(cpu, B, X, Y, update=False)
        g = cpu.download_gradient()
        tol = ABS * max(1.0, float(np.abs(g).max()))
        assert_close(combined.download_gradient(), separate.download_gradient(), REL, tol, what="step %d: combined against separate calls" % step)
        assert_close(combined.download_gradient(), g, REL, tol, what="step %d: combined against the oracle" % step)
        for n in (combined, separate, cpu):
            n.Update_Parameter(B, B)
        wc = cpu.download_parameters()
        combined.upload_parameters(wc)
        separate.upload_parameters(wc)
