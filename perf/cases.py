"""The work this framework is used for, as timed cases: training and inference passes through the network handle.

A training pass is a stretch of an epoch: `steps` mini-batches of a dataset that lies in HBM, each one Forward_Pass,
Compute__Error and the call that joins Backward_Pass, Update_Derivative_Weight and Update_Parameter, then the weights are read
back into a pinned host vector, as a program does that checkpoints or exchanges them.  An inference pass is one Forward_Pass
in the inference state and the read-back of the output layer.

Sizes: the network shapes of bench.py (the reference's own cases among them), the same kinds of network at sizes that are not
multiples of anything, and the small batches that inference sees.
"""
import ctypes
import math

import numpy as np
import torch

from myea_amd import binding as mb
from myea_amd.synthetic import glorot_parameters, simple_debug_layers

# family: layers of the network, head, optimizer and loss - see network()
FAMILIES = ("mlp", "dense", "dense_bn", "residual", "lstm", "bilstm", "lstm_norm", "indrnn")


def _case(name, family, mode, inputs, width, layers, outputs, batch, depth=1, steps=1):
    c = dict(family=family, mode=mode, inputs=inputs, width=width, layers=layers, outputs=outputs, batch=batch, depth=depth, steps=steps)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one request at a time through a small classifier: latency and launches, host buffers on both sides
        _case("infer_mlp_single", "mlp", "infer", 784, 256, 1, 10, batch=1),
        # the reference's CPU-sized network (784-256-10, SGD with momentum): a step is a handful of short launches
        _case("train_mlp_small", "mlp", "train", 784, 256, 1, 10, batch=128, steps=4),
        # a classifier over tabular data: no width is a multiple of 4 and the batch is none either
        _case("train_dense_odd", "dense", "train", 617, 1201, 3, 37, batch=333, steps=4),
        # the wide dense stack of the benchmark (4096 x 4 -> 1000, Adam): the largest contractions and the largest update
        _case("train_dense_wide", "dense", "train", 4096, 4096, 4, 1000, batch=1024, steps=8),
        # eight normalised layers with dropout (Nesterov): contractions of a middle size and a normalisation behind each
        _case("train_dense_bn", "dense_bn", "train", 2048, 2048, 8, 100, batch=512, steps=8),
        # four pre-activation residual blocks at a width and batch half of that
        _case("train_residual", "residual", "train", 1024, 1024, 4, 100, batch=256, steps=4),
        # two LSTM-512 layers over 64 time steps (AMSGrad): the benchmark's recurrent half
        _case("train_lstm", "lstm", "train", 128, 512, 2, 512, batch=256, depth=64, steps=2),
        # a smaller sequence model at sizes of its own: 200 cells, 50 time steps, a batch of 60
        _case("train_lstm_odd", "lstm", "train", 39, 200, 2, 211, batch=60, depth=50, steps=2),
        # both directions of 1024 cells over 512 time steps, a class per step, clipped AdaBound: the longest pass
        _case("train_bilstm", "bilstm", "train", 256, 1024, 1, 32, batch=64, depth=512),
        # the reference's worked example: 27 independently recurrent members in residual blocks over image rows, hundreds of launches
        _case("train_indrnn", "indrnn", "train", 28, 32, 3, 10, batch=256, depth=28, steps=2),
        # LSTM layers normalised inside: every time step is a contraction and its statistics
        _case("train_lstm_norm", "lstm_norm", "train", 64, 256, 2, 256, batch=128, depth=32),
        # a few sequences at a time through a trained recurrent model
        _case("infer_lstm", "lstm", "infer", 128, 512, 2, 512, batch=16, depth=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """over the logarithm of the range; half of them rounded to what people choose, the others as they come"""
    n = _log(rng, lo, hi)
    if rng.random() < 0.5:
        unit = 128 if n >= 512 else 32 if n >= 128 else 8 if n >= 16 else 1
        n = max(lo, min(hi, int(round(n / unit)) * unit))
    return n


_MOST_FLOPS = 1.9e12   # what the two longest listed cases cost


def draw(rng):
    while True:
        family = rng.choice(FAMILIES)
        mode = "infer" if family in ("mlp", "dense", "lstm") and rng.random() < 0.4 else "train"
        steps = 1 if mode == "infer" else 4
        if family == "mlp":
            c = _case("", family, mode, _size(rng, 32, 1024), _size(rng, 32, 1024), rng.randint(1, 3), _size(rng, 2, 100),
                      batch=_size(rng, 1, 64) if mode == "infer" else _size(rng, 16, 512), steps=steps)
        elif family == "dense":
            c = _case("", family, mode, _size(rng, 128, 4096), _size(rng, 256, 4096), rng.randint(2, 5), _size(rng, 10, 1000),
                      batch=_size(rng, 1, 1024) if mode == "infer" else _size(rng, 64, 2048), steps=steps)
        elif family in ("dense_bn", "residual"):
            c = _case("", family, mode, _size(rng, 128, 2048), _size(rng, 128, 2048), rng.randint(2, 8 if family == "dense_bn" else 4),
                      _size(rng, 10, 200), batch=_size(rng, 32, 1024), steps=steps)
        elif family == "lstm":
            width = _size(rng, 64, 1024)   # (the head is at least as wide as the cells below it: what the layout of an LSTM stack's biases takes)
            c = _case("", family, mode, _size(rng, 16, 256), width, rng.randint(1, 2), _size(rng, width, 2 * width),
                      batch=_size(rng, 1, 64) if mode == "infer" else _size(rng, 16, 512), depth=_size(rng, 8, 96), steps=min(steps, 2))
        elif family == "bilstm":
            c = _case("", family, mode, _size(rng, 16, 256), _size(rng, 64, 1024), 1, _size(rng, 8, 64), batch=_size(rng, 16, 128),
                      depth=_size(rng, 16, 192))
        elif family == "lstm_norm":
            width = _size(rng, 32, 384)
            c = _case("", family, mode, _size(rng, 16, 128), width, rng.randint(1, 2), _size(rng, width, 2 * width),
                      batch=_size(rng, 32, 256), depth=_size(rng, 8, 40))
        else:
            c = _case("", family, mode, rng.randint(16, 32), rng.randint(20, 48), 3, 10, batch=_size(rng, 32, 512), depth=_size(rng, 8, 32), steps=2)
        if work(c)["flops"] <= _MOST_FLOPS:
            return c


def network(case):
    """(layers, hyper-parameters) of a case's network"""
    n, L = case["width"], case["layers"]
    # rates at which training neither stands still nor runs away: the gradient is a sum over the batch, and what an Adam step adds to
    # a neuron's sum grows with its fan-in
    adam = dict(adam_learning_rate=min(2e-4, 0.1 / n))
    sgd = dict(type_optimizer_function=mb.OPTIMIZER["GD"], learning_rate=0.02 / case["batch"], learning_momentum=0.9)
    crossentropy, mse = dict(type_loss_function=mb.LOSS["CROSS_ENTROPY"]), dict(type_loss_function=mb.LOSS["MSE"])
    first, head = [dict(units=case["inputs"])], case["outputs"]
    bn = dict(normalization="BATCH_NORMALIZATION")
    drop = dict(dropout="BERNOULLI_INVERTED", keep=0.5)
    family = case["family"]
    if family == "mlp":
        return first + [dict(units=n, activation="TANH")] * L + [dict(units=head, activation="SIGMOID")], dict(sgd, **mse)
    if family == "dense":
        return (first + [dict(units=n, activation="RELU")] * L + [dict(units=head, activation="SOFTMAX")],
                dict(type_optimizer_function=mb.OPTIMIZER["ADAM"], **adam, **crossentropy))
    if family == "dense_bn":
        return (first + [dict(units=n, activation="RELU", **bn, **drop)] * L + [dict(units=head, activation="SOFTMAX")],
                dict(sgd, use_Nesterov=1, **crossentropy))
    if family == "residual":
        block = [dict(type="residual", block_depth=2), dict(units=n, activation="RELU", **bn), dict(units=n, activation="RELU", **bn, **drop)]
        return (first + [dict(units=n, activation="RELU")] + block * L + [dict(units=head, activation="SOFTMAX")],
                dict(sgd, learning_rate=0.1 * sgd["learning_rate"], **crossentropy))   # (the sums of un-normalised shortcuts grow with the depth)
    if family == "lstm":
        return (first + [dict(type="lstm", units=n)] * L + [dict(units=head, activation="LINEAR")],
                dict(type_optimizer_function=mb.OPTIMIZER["AMSGRAD"], **adam, **mse))
    if family == "bilstm":
        return (first + [dict(type="lstm", units=n, bidirectional=True)] * L + [dict(units=head, activation="SOFTMAX")],
                dict(type_optimizer_function=mb.OPTIMIZER["ADABOUND"], use_clip_gradient=1, clip_gradient=1.0, **adam, **crossentropy))
    if family == "lstm_norm":
        return (first + [dict(type="lstm", units=n, **bn)] * L + [dict(units=head, activation="LINEAR")],
                dict(type_optimizer_function=mb.OPTIMIZER["ADAM"], **adam, **mse))
    return (simple_debug_layers(inputs=case["inputs"], outputs=head, units=n, blocks_per_group=L),   # indrnn
            dict(type_optimizer_function=mb.OPTIMIZER["AMSGRAD"], **adam, **crossentropy, regularization__max_norm_constraints=8.0,
                 normalization_momentum_average=1.0, normalization_epsilon=0.1, number_time_delays=case["depth"] - 1))


def _describe(case):
    layers, hyper = network(case)
    return mb.make_desc(layers, case["batch"], case["depth"]), hyper


def prepare(case, seed):
    """The network with its weights on the device, a dataset of `steps` mini-batches in HBM (a single request: on the host) and the
    host vector that results are read into."""
    desc, hyper = _describe(case)
    B, T, steps = case["batch"], case["depth"], case["steps"]
    train = case["mode"] == "train"
    net = mb.HipNetwork(desc, mb.default_hyper(**hyper))
    net.set_stream(torch.cuda.current_stream().cuda_stream)
    net.set_state_propagation(mb.STATE_TRAINING if train else mb.STATE_INFERENCE)
    net.upload_parameters(glorot_parameters(desc, seed))
    net.Clear_Training_Arrays()
    rng = np.random.default_rng(seed + 1)
    if train and desc.total_mask_units:
        net.upload_masks((rng.random(desc.total_mask_units) < 0.5).astype(np.uint8))
    examples, n_in, n_out = B * steps, case["inputs"], case["outputs"]
    if case["family"] in ("mlp", "indrnn"):   # pixels
        X = rng.random((examples, T * n_in), dtype=np.float32)
    else:
        X = rng.standard_normal((examples, T * n_in), dtype=np.float32)
    state = dict(case=case, net=net, host=not train and case["family"] == "mlp")
    state["x"] = X if state["host"] else torch.from_numpy(X).cuda()
    if train:
        if case["family"] in ("lstm", "lstm_norm"):   # a target per time step
            Y = rng.standard_normal((examples, T * n_out), dtype=np.float32)
        else:                                         # a class per example or time step
            Y = np.zeros((examples * T, n_out), dtype=np.float32)
            Y[np.arange(examples * T), rng.integers(0, n_out, examples * T)] = 1.0
            Y = Y.reshape(examples, T * n_out)
        state["y"] = torch.from_numpy(Y).cuda()
        state["out"] = torch.empty(desc.total_parameters, dtype=torch.float32, pin_memory=True)
    else:
        state["out"] = torch.empty(T, B, n_out, dtype=torch.float32, pin_memory=True)
    return state


def run(state):
    case, net, x, out = state["case"], state["net"], state["x"], state["out"]
    B = case["batch"]
    destination, count = ctypes.c_void_p(out.data_ptr()), out.numel()
    if case["mode"] == "infer":
        net.Forward_Pass(B, x, on_device=not state["host"])
        net._check(net.lib.myea_hip_download_tensor(net.handle, net.desc.n_layers - 1, mb.TENSOR["OUTPUTS"], destination, count))
        return out
    y = state["y"]
    for first in range(0, B * case["steps"], B):
        net.Forward_Pass(B, x[first:first + B], on_device=True)
        net.Compute__Error(B, y[first:first + B], on_device=True)
        net.Backward_Pass__Update_Derivative_Weight__Update_Parameter(B, B)
    net._check(net.lib.myea_hip_download_parameters(net.handle, destination, count))
    return out


def work(case):
    """Products of forward, delta and weight gradient (an LSTM cell: four gate rows, recurrent products at T - 1 steps); bytes: inputs
    and targets, the weights (read and written by a step) and the optimizer's vectors."""
    desc, hyper = _describe(case)
    lib = mb.load_library()
    B, T, steps = case["batch"], case["depth"], case["steps"]
    forward = delta = 0.0
    for i in range(1, desc.n_layers):
        l = desc.layers[i]
        if l.type_layer in (mb.LAYER_RESIDUAL, mb.LAYER_AVERAGE_POOLING, mb.LAYER_MAX_POOLING):
            continue
        below = lib.myea_net_desc_previous_layer(ctypes.byref(desc), i)
        fan_in, width = (int(lib.myea_net_desc_number_outputs(ctypes.byref(desc), j)) for j in (below, i))
        if l.type_layer == mb.LAYER_LSTM:
            directions = 2 if l.use_bidirectional else 1
            product, recurrent = 8.0 * directions * B * T * width * fan_in, 8.0 * directions * B * (T - 1) * width * width
        else:
            product, recurrent = 2.0 * B * T * width * fan_in, 0.0
        forward += product + recurrent
        delta += recurrent + (product if below else 0.0)
    P, data = int(desc.total_parameters), B * T * (case["inputs"] + case["outputs"])
    if case["mode"] == "infer":
        return {"bytes": 4.0 * (P + data), "flops": forward}
    vectors = {"GD": 1, "ADAM": 2, "AMSGRAD": 3, "ADABOUND": 2}[next(k for k, v in mb.OPTIMIZER.items() if v == hyper["type_optimizer_function"])]
    return {"bytes": 4.0 * steps * (P * (2 + 2 * vectors) + data), "flops": steps * (2 * forward + delta)}


def tolerance(case):
    """About four times what the weights move, after two passes, when every example of a mini-batch stands at another place and its
    inputs carry a last-bit error - another order of the sums, and what that does to ReLUs at zero and to Adam's steps where a
    gradient is rounding noise - over the listed and some 90 drawn cases; for inference, four times the distance from the serial
    sums of the CPU oracle."""
    if case["mode"] == "infer":
        return {"rel": 3e-6, "max": 2e-5}
    rel, most = {"mlp": (1.5e-7, 1.5e-6), "dense": (2.5e-3, 0.09), "dense_bn": (3e-4, 0.015), "residual": (2e-5, 2e-3), "lstm": (2e-5, 0.02),
                 "bilstm": (1e-7, 1e-5), "indrnn": (8e-4, 0.02), "lstm_norm": (5e-5, 0.02)}[case["family"]]
    return {"rel": rel, "max": most}
