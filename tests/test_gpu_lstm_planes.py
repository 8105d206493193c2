"""The LSTM time loops on the BF16 matrix cores (16 .. 512 cells, any width) where they can go wrong: an odd number of members (half a
block of k's without an owner), one member, a last member of one cell, one and several row tiles per group, a last group with fewer of
them, examples missing from the last tile, more steps than the exchange buffer has slots, two directions, zoneout, a smaller batch
behind a larger one - against one launch per time step (MYEA_LSTM_RESIDENT=0; the two paths sum in another order and round their gate
functions differently by a few ulp: rel 1e-4 / abs 1e-5 as for the other LSTM paths) - and what the planes cannot hold."""
import ctypes as C

import numpy as np
import pytest
import torch

from myea_amd import binding as mb
from tests.common import assert_close, environment, run_step
from tests.test_gpu_lstm_resident import ABS, REL, _compare, _loop_launches, _net, _setup, lstm, planes_plan, zone

pytestmark = pytest.mark.gpu

# cells, two directions, zoneout, T, B, Bmax
CASES = [(16, False, False, 9, 1, 1), (17, False, False, 5, 16, 16), (47, False, False, 6, 17, 20), (257, True, False, 6, 33, 40),
         (200, False, True, 7, 60, 60), (256, False, False, 5, 520, 520), (512, False, True, 6, 129, 136), (511, True, False, 5, 70, 70),
         (500, False, False, 5, 300, 300), (64, True, True, 12, 3, 4)]


@pytest.mark.parametrize("cells,both,zoned,T,B,Bmax", CASES)
def test_loop_of_any_width(cells, both, zoned, T, B, Bmax):
    specs = [dict(units=7), (zone if zoned else lstm)(cells, **(dict(bidirectional=True) if both else {})), dict(units=cells, activation="LINEAR")]
    desc, h, w, masks, X, Y = _setup(specs, T, B, Bmax, seed=cells)
    loop, steps = _net(desc, h, w, masks), _net(desc, h, w, masks)
    for b in (B, (B + 1) // 2):
        with environment(MYEA_LSTM_RESIDENT="0"):
            steps.Clear_Training_Arrays()
            run_step(steps, b, X[:b], Y[:b], update=False)
        loop.Clear_Training_Arrays()
        loop.profile_enable(True)
        run_step(loop, b, X[:b], Y[:b], update=False)
        launches = _loop_launches(loop)
        loop.profile_enable(False)
        assert launches == (1, 1), "the time loops did not run as one launch each"
        _compare(desc, loop, steps, b, T, "%d examples" % b)


# the last batch of the backward loop and the first of one launch a step, where the forward pass stays a loop; the first batch without either
LINES = [(16, False, 32768, 32769, None), (100, False, 4096, 4097, 8193), (256, False, 1280, 1281, None), (480, False, 512, 513, None), (500, False, 768, 769, 3713),
         (200, True, 768, 769, None), (224, True, 640, 641, None), (448, True, 192, 193, None)]


@pytest.mark.parametrize("cells,both,loop,beyond,without", LINES)
def test_lines_between_the_backward_loop_and_one_launch_a_step(cells, both, loop, beyond, without):
    """values of both passes and the gradient against one launch a step throughout"""
    T, directions = 3, 2 if both else 1
    specs = [dict(units=3), lstm(cells, **(dict(bidirectional=True) if both else {})), dict(units=cells, activation="LINEAR")]
    launches = {loop: (1, 1), beyond: (1, directions * (T - 1)), without: (directions * (T - 1),) * 2}
    Bmax = without or beyond
    desc, h, w, masks, X, Y = _setup(specs, T, Bmax, Bmax, seed=cells)
    net, steps = _net(desc, h, w, masks), _net(desc, h, w, masks)
    for B in sorted((b for b in launches if b), reverse=True):
        with environment(MYEA_LSTM_RESIDENT="0"):
            steps.Clear_Training_Arrays()
            run_step(steps, B, X[:B], Y[:B], update=False)
        net.Clear_Training_Arrays()
        net.profile_enable(True)
        run_step(net, B, X[:B], Y[:B], update=False)
        assert _loop_launches(net) == launches[B], "%d examples" % B
        net.profile_enable(False)
        _compare(desc, net, steps, B, T, "%d examples" % B)


@pytest.mark.parametrize("dirs", [1, 2])
def test_every_plan_fits_the_buffers_of_a_larger_batch(dirs):
    lib = mb.load_library()
    floats = [getattr(lib, "_ZN4myea%sEmmi" % n) for n in ("27lstm_planes_exchange_floats", "25lstm_planes_shares_floats")]
    for f in floats:
        f.argtypes, f.restype = [C.c_size_t, C.c_size_t, C.c_int], C.c_size_t
    for cells in (16, 17, 40, 100, 128, 129, 200, 224, 256, 257, 300, 320, 352, 448, 480, 500, 512):
        largest, plans = [0, 0], 0
        for B in sorted(set(list(range(1, 600)) + [n * 16 + d for n in range(40, 600, 7) for d in (0, 1, 15)] + [2 ** n + d for n in range(10, 17) for d in (0, 1)])):
            plan = planes_plan(cells, B, dirs)
            if plan.ok:
                tiles = dirs * plan.row_groups * plan.rs
                plans += 1
                largest[0] = max(largest[0], tiles * ((cells + 31) // 32) * 3072 * 4 // 4)
                if plan.backward:
                    largest[1] = max(largest[1], tiles * 2 * plan.members ** 2 * 256)
            for f, most in zip(floats, largest):
                assert f(cells, B, dirs) >= most, (cells, B)
        assert plans > 100 and min(largest) > 0


@pytest.mark.parametrize("cells,B", [(40, 20), (300, 200)])
def test_weights_beyond_the_planes(cells, B):
    """Recurrent weights of 2^110 next to ordinary ones: the planes of such a weight are an infinity and NaNs, so every sum it is part of
    is computed again; forward, the gates saturate (or not, where a weight meets an h of zero) as with one launch per step; backward, the
    share of a member that holds one is finite or an infinity as there."""
    T = 4
    specs = [dict(units=5), lstm(cells), dict(units=cells, activation="LINEAR")]
    desc, h, w, masks, X, Y = _setup(specs, T, B, B, seed=3)
    layer = desc.layers[1]
    rng = np.random.default_rng(5)
    at = rng.choice(np.arange(layer.first_connection_index, layer.last_connection_index), 40, replace=False)
    for value in (2.0 ** 110, np.inf):
        v = w.copy()
        v[at] = np.float32(value)
        out = []
        for resident in ("1", "0"):
            net = _net(desc, h, v, masks)
            with environment(MYEA_LSTM_RESIDENT=resident):
                net.Forward_Pass(B, X)
                out.append(net.download_tensor(1, mb.TENSOR["OUTPUTS"], T * B * cells).copy())
                if np.isfinite(value):
                    net.Compute__Error(B, Y)
                    net.Backward_Pass(B)
                    out[-1] = (out[-1], net.download_tensor(1, mb.TENSOR["ERRORS"], T * B * cells).copy())
                else:
                    out[-1] = (out[-1],)
        for a, b in zip(*out):
            same = np.isfinite(a) & np.isfinite(b)
            assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~same], b[~same], equal_nan=True)
            assert (np.abs(b[same]) < 1e3).any()   # ordinary values among them are held to the ordinary tolerance
            assert_close(a[same], b[same], REL, ABS, what="weights of %g" % value)


def test_two_networks_on_two_streams_take_turns():
    """each loop fills the device by itself: launched side by side, their workgroups would wait for compute units the other's hold"""
    T, B, cells = 24, 256, 500
    specs = [dict(units=5), lstm(cells), dict(units=cells, activation="LINEAR")]
    desc, h, w, masks, X, Y = _setup(specs, T, B, B, seed=11)
    nets = [_net(desc, h, w, masks) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    x, y = torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda()
    torch.cuda.synchronize()
    for n, s in zip(nets, streams):
        n.set_stream(s.cuda_stream)
    for _ in range(6):
        for n in nets:
            n.Clear_Training_Arrays()
            n.Forward_Pass(B, x, on_device=True)
            n.Compute__Error(B, y, on_device=True)
            n.Backward_Pass(B)
    for n in nets:
        n.synchronize()   # a wait that gave up is reported here
    a, b = (n.download_tensor(1, mb.TENSOR["ERRORS"], T * B * cells) for n in nets)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("switches", [dict(), dict(MYEA_LSTM_BACKWARD_SETS="0"),
                                      dict(MYEA_LSTM_BACKWARD_SETS="0", MYEA_LSTM_RESIDENT_TEST_NEVER_EARLY="1")], ids=["sets", "one-stream", "one-stream-late"])
def test_512_cells_beyond_a_row_tile_per_group(switches):
    """where the backward pass is the FP32 loop's: both of its forms behind this forward loop, with a ragged last group"""
    T, B, cells = 5, 141, 512
    specs = [dict(units=7), lstm(cells), dict(units=cells, activation="LINEAR")]
    desc, h, w, masks, X, Y = _setup(specs, T, B, 150, seed=17)
    loop, steps = _net(desc, h, w, masks), _net(desc, h, w, masks)
    with environment(MYEA_LSTM_RESIDENT="0"):
        run_step(steps, B, X, Y, update=False)
    with environment(**switches):
        loop.profile_enable(True)
        run_step(loop, B, X, Y, update=False)
        assert _loop_launches(loop) == (1, 1)
    _compare(desc, loop, steps, B, T, "512 cells")
