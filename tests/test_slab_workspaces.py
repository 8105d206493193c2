"""Slabs of the split-k weight gradients against the workspace that holds them: the number of slabs is no monotone function of the
rows (from 4096 rows on a slab is deeper; the narrow kernel halves its workgroups beyond 32768 rows), so the workspace of a
network's largest batch has to hold what a smaller batch writes."""
import ctypes as C

import numpy as np
import pytest
import torch

from myea_amd import binding as mb
from tests.common import assert_close, glorot_parameters
from tests.oracle_lib import OracleNetwork


def _function(name, *kinds):
    f = getattr(mb.load_library(), name)
    f.argtypes, f.restype = kinds, C.c_int
    return f


@pytest.mark.parametrize("M,N", [(1, 1), (64, 64), (65, 64), (40, 200), (256, 256), (256, 784), (512, 512), (1000, 37), (1024, 512), (2048, 1000), (4096, 4096)])
def test_split_k_never_exceeds_its_bound(M, N):
    count, most = (_function("_ZN4myea%sEiii" % n, C.c_int, C.c_int, C.c_int) for n in ("12gemm_split_k", "17gemm_split_k_most"))
    reached, ks = 0, list(range(1, 700)) + list(range(700, 20000, 53)) + [4063, 4064, 4065, 4095, 4096, 4097, 16383, 16384, 100000, 10 ** 7, 2 ** 31 - 1]
    for k in sorted(ks):
        assert count(M, N, k) >= 1, k
        reached = max(reached, count(M, N, k))
        assert reached <= most(M, N, k), k
    assert most(M, N, 2 ** 31 - 1) <= 32


def test_narrow_kernel_never_exceeds_its_bound():
    count, most = (_function("_ZN4myea%sEmmm" % n, C.c_size_t, C.c_size_t, C.c_size_t) for n in ("15narrow_dw_slabs", "20narrow_dw_slabs_most"))
    assert count(32, 32, 32768) == 128 and count(32, 32, 32769) == 65
    reached = 0
    for rows in list(range(1, 5000)) + list(range(5000, 140000, 61)) + [10 ** 6, 10 ** 8]:
        reached = max(reached, count(27, 28, rows))
        assert reached <= most(27, 28, rows), rows


def test_buffers_of_the_time_loops_end_where_the_loops_do():
    """sizes at any batch beyond the last plan: 8 groups of 4 tiles, two steps of 30 x 30 KiB each, at 480 cells, one tile a group at 512"""
    shares, exchange = getattr(mb.load_library(), "_ZN4myea25lstm_planes_shares_floatsEmmi"), getattr(mb.load_library(), "_ZN4myea27lstm_planes_exchange_floatsEmmi")
    for f in (shares, exchange):
        f.argtypes, f.restype = [C.c_size_t, C.c_size_t, C.c_int], C.c_size_t
    for B in (4096, 16384, 10 ** 6):
        assert shares(480, B, 1) == 8 * 4 * 2 * 30 * 30 * 256 and shares(512, B, 1) == shares(512, B, 2) == 8 * 2 * 32 * 32 * 256
        assert exchange(480, B, 1) <= 8 * 29 * 15 * 3072
    assert max(f(c, 10 ** 7, d) for f in (shares, exchange) for c in range(16, 513) for d in (1, 2)) <= 2 ** 25   # 128 MiB


def _gradients(specs, Bmax, T, B, seed):
    desc = mb.make_desc(specs, Bmax, T)
    h = mb.default_hyper(type_optimizer_function=mb.OPTIMIZER["ADAM"], type_loss_function=mb.LOSS["MSE"])
    rng = np.random.default_rng(seed)
    X, Y = (rng.normal(0, 1, (B, T * s["units"])).astype(np.float32) for s in (specs[0], specs[-1]))
    w, out = glorot_parameters(desc, seed), []
    for n in (mb.HipNetwork(desc, h), OracleNetwork(desc, h, threads=8)):
        n.set_state_propagation(mb.STATE_TRAINING)
        n.upload_parameters(w)
        n.Clear_Training_Arrays()
        n.Forward_Pass(B, X)
        n.Compute__Error(B, Y)
        n.Backward_Pass(B)
        n.Update_Derivative_Weight(B, 1, desc.n_layers)
        out.append(n.download_gradient())
    got, want = out
    # a gradient is a sum over the rows: both sides' rounding grows with its largest terms
    assert_close(got, want, 1e-4, 1e-5 * max(1.0, float(np.abs(want).max())), what="gradient, %d of %d rows" % (B, Bmax))


@pytest.mark.gpu
@pytest.mark.parametrize("layers,Bmax,batches", [
    ((256, 256), 5000, (3000, 5000)),      # 16 slabs at 3000 rows, 4 at 5000
    ((784, 256), 4096, (4095, 4096)),      # 5 and 4
    ((28, 32), 32769, (32768, 32769)),     # the narrow kernel: 128 and 65
], ids=["256x256", "256x784", "narrow"])
def test_smaller_batch_with_more_slabs(layers, Bmax, batches):
    for B in batches:
        _gradients([dict(units=layers[0]), dict(units=layers[1], activation="LINEAR")], Bmax, 1, B, 7)


@pytest.mark.gpu
def test_small_lstm_over_many_rows():
    """Four gates of 16 cells over 32 inputs are one 64 x 64 tile: 18 slabs over 2 x 2304 rows."""
    _gradients([dict(units=32), dict(type="lstm", units=16), dict(units=16, activation="LINEAR")], 2304, 2, 2304, 5)


@pytest.mark.gpu
def test_call_without_allocations_sizes_its_pieces_for_the_batch():
    """16 slabs at 3000 rows, 4 at 5000, in front of a second layer whose LSTM slabs lie behind them: bit for bit the ordinary call."""
    from tests.test_zz_no_alloc import _gradients as both
    desc = mb.make_desc([dict(units=256), dict(units=256, activation="TANH"), dict(type="lstm", units=16), dict(units=16, activation="LINEAR")], 5000)
    net = mb.HipNetwork(desc, mb.default_hyper(type_optimizer_function=mb.OPTIMIZER["ADAM"], type_loss_function=mb.LOSS["MSE"]))
    net.set_state_propagation(mb.STATE_TRAINING)
    net.upload_parameters(glorot_parameters(desc, 9))
    rng = np.random.default_rng(9)
    for B in (5000, 3000):
        X, Y = (rng.normal(0, 1, (B, n)).astype(np.float32) for n in (256, 16))
        got, want = both(net, B, X, Y)
        assert np.abs(want).max() > 0 and np.array_equal(got, want)


@pytest.mark.gpu
def test_batches_of_other_sizes_share_the_table_of_narrow_layers():
    """The table of narrow layers that lies on the device holds for any number of rows of as many slabs (8 at 1793 .. 2048): a batch of
    another size neither waits for the stream - which a capture would refuse - nor sums other rows than its own."""
    Bmax, sizes = 2048, (2048, 1800, 2047)
    desc = mb.make_desc([dict(units=28), dict(units=32, activation="TANH"), dict(units=17, activation="TANH"), dict(units=10, activation="LINEAR")], Bmax)
    h = mb.default_hyper(type_optimizer_function=mb.OPTIMIZER["ADAM"], type_loss_function=mb.LOSS["MSE"])
    gpu, cpu = mb.HipNetwork(desc, h), OracleNetwork(desc, h, threads=8)
    rng = np.random.default_rng(3)
    X, Y = (rng.normal(0, 1, (Bmax, n)).astype(np.float32) for n in (28, 10))
    w = glorot_parameters(desc, 3)
    for n in (gpu, cpu):
        n.set_state_propagation(mb.STATE_TRAINING)
        n.upload_parameters(w)
    stream = torch.cuda.Stream()
    gpu.set_stream(stream.cuda_stream)
    for B in sizes:
        for n in (gpu, cpu):
            n.Clear_Training_Arrays()
            n.Forward_Pass(B, X[:B])
            n.Compute__Error(B, Y[:B])
            n.Backward_Pass(B)
        cpu.Update_Derivative_Weight(B, 1, desc.n_layers)
        want = cpu.download_gradient()
        if B == sizes[0]:
            gpu.Update_Derivative_Weight(B, 1, desc.n_layers)
            assert_close(gpu.download_gradient(), want, 1e-4, 1e-5 * float(np.abs(want).max()), what="gradient of %d examples" % B)
            continue
        gpu.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            gpu.Update_Derivative_Weight(B, 1, desc.n_layers)
        for replay in range(1, 4):   # each adds the gradient once more
            graph.replay()
            torch.cuda.synchronize()
            assert_close(gpu.download_gradient(), replay * want, 1e-4, 1e-5 * replay * float(np.abs(want).max()), what="gradient of %d examples, replay %d" % (B, replay))
