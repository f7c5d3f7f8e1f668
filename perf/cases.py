"""The work a program hands to this framework, as cases whose time can be measured.

Every case is one pass through the public entry points: a training step (`Replica.step`), an epoch over a partition that
lies on the device (`Replica.train_epoch`), a prediction (`Replica.forward`), the flat optimizer update
(`Context.optimizer_update`) or the averaging of partitions' replicas (`average_replicas`).  Sizes are those of the
repository's own configurations, and generic ragged ones between them: batch sizes, features and units that are no
multiples of anything, colour images, layers stacked on layers.
"""
import math

import numpy as np
import torch

import scanet3_amd as S
from scanet3_amd import _lib as L

ACTIVATIONS = {"sigmoid": S.Sigmoid, "tanh": S.Tanh, "relu": S.ReLU()}
OPTIMIZERS = {"SGD": lambda: S.SGD(0.01, 0.9), "AdaGrad": lambda: S.AdaGrad(0.001), "AdaDelta": lambda: S.AdaDelta(),
              "RMSProp": lambda: S.RMSProp(0.001), "Adam": lambda: S.Adam(0.001), "Nadam": lambda: S.Nadam(),
              "Adamax": lambda: S.Adamax(0.001), "AMSGrad": lambda: S.AMSGrad(0.001)}
_context = []


def context():
    """The one context a program keeps for its device."""
    if not _context:
        _context.append(S.Context(0))
    return _context[0]


class View:
    """float32 device memory of the library as something `torch.as_tensor` reads; keeps its owner alive."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": "<f4", "data": (int(ptr), False), "version": 3, "strides": None}


def view(owner, ptr, n):
    return torch.as_tensor(View(owner, ptr.value, n), device="cuda")


class Handles:
    """A model with its replicas, given back when the last reference goes."""

    def __init__(self, layers, loss, in_shape, batch, alg, flags=0, replicas=1):
        self.model = S.CompiledModel(context(), [l.desc() for l in layers.layers], loss.kind, in_shape, batch, flags)
        self.replicas = [self.model.replica(alg) for _ in range(replicas)]

    def __del__(self):
        for r in self.replicas:
            r.close()
        self.model.close()


class Buffers:
    """Flat device vectors of one length."""

    def __init__(self, count, n):
        self.items = [context().alloc(n) for _ in range(count)]

    def __del__(self):
        for b in self.items:
            b.free()


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


# ---------------------------------------------------------------------------------------------------------------- models


def layers_of(case):
    kind = case["kind"]
    if kind == "mlp":
        widths = [case[k] for k in ("hidden1", "hidden2", "hidden3") if case.get(k)]
        model = None
        for w in widths:
            layer = S.Dense(w, ACTIVATIONS[case["activation"]])
            model = layer if model is None else model >> layer
        return model >> S.Dense(case["classes"], S.Softmax)
    if kind == "cnn":
        pad = S.Same if case["padding"] == "same" else S.Valid
        model = S.Conv2D(case["filters1"], padding=pad, activation=S.ReLU())
        if case["batchnorm"]:
            model = model >> S.BatchNorm(fused=True)
        stride = (case["pool_stride"],) * 2
        model = model >> S.Pool2D(strides=stride) >> S.Conv2D(case["filters2"], padding=pad, activation=S.ReLU()) >> S.Pool2D(strides=stride)
        model = model >> S.Flatten
        if case["hidden"]:
            model = model >> S.Dense(case["hidden"], S.ReLU())
        return model >> S.Dense(case["classes"], S.Softmax)
    cell = S.LSTM if case["cell"] == "lstm" else S.SimpleRNN
    model = cell(case["units1"], returnSequence=bool(case["units2"]))
    if case["units2"]:
        model = model >> cell(case["units2"])
    return model >> S.Dense(1, S.Tanh)


def in_shape_of(case):
    if case["kind"] == "mlp":
        return (case["features"],)
    if case["kind"] == "cnn":
        return (case["side"], case["side"], case["channels"])
    return (case["steps"], case["features"])


def initialise(weights, params, g):
    """The layers' default initializers: Glorot-uniform kernels, orthogonal recurrent weights, zero biases (one for an LSTM's
    forget gate), ones where a BatchNorm starts from one."""
    weights.zero_()
    for path, shape, offset in params:
        leaf = path.rsplit("/", 1)[-1]
        n = int(np.prod(shape))
        part = weights[offset:offset + n]
        if leaf in ("gamma", "moving_variance") or "forget/1/" in path:
            part.fill_(1.0)
        elif leaf == "recurrent_weights":
            q, r = torch.linalg.qr(torch.randn(shape, generator=g, device="cuda"))
            part.copy_((q * torch.sign(torch.diagonal(r))).flatten())
        elif leaf not in ("beta", "moving_mean") and len(shape) > 1:
            limit = math.sqrt(6.0 / (int(np.prod(shape[:-1])) + shape[-1]))
            part.uniform_(-limit, limit, generator=g)


def batch_of(case, rows, g):
    """Images and pixel vectors are uniform in [0, 1), other features N(0, 1); labels one-hot, targets uniform in [-1, 1)."""
    shape = (rows,) + in_shape_of(case)
    if case["kind"] == "cnn" or (case["kind"] == "mlp" and case["inputs"] == "pixels"):
        x = torch.rand(shape, generator=g, device="cuda")
    else:
        x = torch.randn(shape, generator=g, device="cuda")
    if case["kind"] == "recurrent":
        return x, torch.rand((rows, 1), generator=g, device="cuda") * 2 - 1
    labels = torch.randint(0, case["classes"], (rows,), generator=g, device="cuda")
    return x, torch.nn.functional.one_hot(labels, case["classes"]).float()


def prepare_model(case, seed):
    g = generator(seed)
    flags = L.FLAG_GEMM_BF16 if case.get("dtype") == "bf16" else 0
    loss = S.MeanSquaredError if case["kind"] == "recurrent" else S.CategoricalCrossentropy
    alg = None if case["call"] == "predict" else S.Adam(case["rate"])
    handles = Handles(layers_of(case), loss, in_shape_of(case), case["batch"], alg, flags)
    replica = handles.replicas[0]
    weights = view(handles, *replica.flat(-2))
    initialise(weights, handles.model.params, g)
    replica.flat(-2)  # the weights were written through the view
    x, y = batch_of(case, case["batch"] * case.get("batches", 1), g)
    # training goes on from a state that some thousand steps have left: the running mean square of every gradient is
    # there (a first step from zeros moves a weight by the sign of its gradient, however small that is)
    state = {"case": case, "handles": handles, "replica": replica, "x": x, "y": y, "iteration": 5000}
    if alg is not None:
        state["outputs"] = {"weights": weights, "gradients": view(handles, *replica.flat(-1)), "momentum": view(handles, *replica.flat(0)),
                            "velocity": view(handles, *replica.flat(1))}
        state["outputs"]["velocity"].uniform_(0.5e-4, 1.5e-4, generator=g)
    return state


def prepare(case, seed):
    if case["kind"] == "optimizer":
        g, n = generator(seed), case["n"]
        states = len(S.dsl.STATE_NAMES[OPTIMIZERS[case["optimizer"]]().kind])
        buffers = Buffers(2 + states, n)
        views = [view(buffers, b.ptr, n) for b in buffers.items]
        views[0].normal_(0.0, 0.02, generator=g)
        views[1].normal_(0.0, 1e-3, generator=g)
        for v in views[2:]:  # squares and running means of gradients: small and not negative
            v.uniform_(0.0, 1e-6, generator=g)
        state = {"case": case, "buffers": buffers, "alg": OPTIMIZERS[case["optimizer"]](), "iteration": 0, "outputs": [views[0]] + views[2:]}
    elif case["kind"] == "average":
        g = generator(seed)
        layers = S.Dense(case["hidden"], S.ReLU()) >> S.Dense(case["classes"], S.Softmax)
        handles = Handles(layers, S.CategoricalCrossentropy, (case["features"],), 8, S.Adam(0.001), 0, case["replicas"])
        outputs = []
        for r in handles.replicas:
            outputs.append([view(handles, *r.flat(slot)) for slot in (-2, 0, 1)])
            outputs[-1][0].normal_(0.0, 0.02, generator=g)
            outputs[-1][1].normal_(0.0, 1e-3, generator=g)
            outputs[-1][2].uniform_(0.0, 1e-6, generator=g)
        state = {"case": case, "handles": handles, "outputs": outputs}
    else:
        state = prepare_model(case, seed)
    torch.cuda.synchronize()  # the inputs were made on torch's stream, the library has its own
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "optimizer":
        state["iteration"] += 1
        b = state["buffers"].items
        context().optimizer_update(state["alg"], b[0], b[1], b[2:], state["iteration"])
        return state["outputs"]
    if case["kind"] == "average":
        S.average_replicas(state["handles"].replicas)
        return state["outputs"]
    replica, x, y = state["replica"], state["x"].data_ptr(), state["y"].data_ptr()
    if case["call"] == "predict":
        return replica.forward(x)
    if case["call"] == "epoch":
        done, loss = replica.train_epoch(x, y, case["batch"] * case["batches"], case["batch"], state["iteration"])
        state["iteration"] += done
        return dict(state["outputs"], loss=loss)
    state["iteration"] += 1
    replica.step(x, y, state["iteration"])
    return state["outputs"]


# ----------------------------------------------------------------------------------------------------------- work, limits


def conv_size(size, kernel, stride, padding):
    return -(-size // stride) if padding == "same" else -(-(size - kernel + 1) // stride)


def cnn_sizes(case):
    """Side lengths behind conv 1, pool 1, conv 2, pool 2."""
    a = conv_size(case["side"], 3, 1, case["padding"])
    b = conv_size(a, 2, case["pool_stride"], "valid")
    c = conv_size(b, 3, 1, case["padding"])
    return a, b, c, conv_size(c, 2, case["pool_stride"], "valid")


def step_work(case):
    """(flops of a forward pass, flops of the gradients, weights) of one batch; element-wise work is not counted."""
    B = case["batch"]
    forward = backward = weights = 0
    products = []  # (flops forward, the layer's input gradient is needed)
    if case["kind"] == "mlp":
        widths = [case["features"]] + [case[k] for k in ("hidden1", "hidden2", "hidden3") if case.get(k)] + [case["classes"]]
        for a, b in zip(widths, widths[1:]):
            products.append(2.0 * B * a * b)
            weights += a * b + b
    elif case["kind"] == "cnn":
        a, _, c, d = cnn_sizes(case)
        f1, f2 = case["filters1"], case["filters2"]
        products += [2.0 * B * a * a * 9 * case["channels"] * f1, 2.0 * B * c * c * 9 * f1 * f2]
        widths = [d * d * f2] + ([case["hidden"]] if case["hidden"] else []) + [case["classes"]]
        weights += 9 * case["channels"] * f1 + 9 * f1 * f2 + (4 * f1 if case["batchnorm"] else 0)
        for m, n in zip(widths, widths[1:]):
            products.append(2.0 * B * m * n)
            weights += m * n + n
    else:
        gates, features = (4 if case["cell"] == "lstm" else 1), case["features"]
        for h in [case["units1"]] + ([case["units2"]] if case["units2"] else []):
            products.append(2.0 * B * case["steps"] * gates * h * (features + h))
            weights += gates * (features + h + 1) * h
            features = h
        products.append(2.0 * B * features)
        weights += features + 1
    forward = sum(products)
    backward = 2 * forward - products[0]  # every layer's weight gradient, and its input gradient but for the first layer's
    if case["kind"] == "recurrent":
        backward += products[0] * case["units1"] / (case["features"] + case["units1"])  # ... the first recurrence still carries its state back
    return forward, backward, weights


def work(case):
    if case["kind"] == "optimizer":
        states = len(S.dsl.STATE_NAMES[OPTIMIZERS[case["optimizer"]]().kind])
        return {"bytes": 4.0 * case["n"] * (3 + 2 * states), "flops": 10.0 * case["n"]}
    if case["kind"] == "average":
        n = (case["features"] + 1) * case["hidden"] + (case["hidden"] + 1) * case["classes"]
        return {"bytes": 3.0 * 4 * n * 2 * case["replicas"], "flops": 3.0 * n * case["replicas"]}
    forward, backward, weights = step_work(case)
    outputs = case.get("classes", 1)
    rows = case["batch"] * case.get("batches", 1)
    data = 4.0 * rows * (int(np.prod(in_shape_of(case))) + outputs)
    if case["call"] == "predict":
        return {"bytes": data + 4.0 * weights, "flops": forward}
    passes = case.get("batches", 1)
    return {"bytes": data + 4.0 * weights * 7 * passes, "flops": (forward + backward) * passes}  # weights and two states in and out, gradients out


def tolerance(case):
    """About four times what the outputs of one and of three steps move by when every input and weight is off by one
    rounding and the rows of the batch come in another order (the largest of some 250 drawn cases of each kind).  Where a
    ReLU or a maximum sits, a value within a rounding of its kink may land on the other side and take its whole gradient
    with it; a simple recurrence without a squashing function multiplies a rounding by its weights at every time step."""
    if case["kind"] in ("optimizer", "average"):
        return {"rel": 1e-6}
    if case["call"] == "predict":
        return {"rel": 1e-5}
    if case["kind"] == "cnn":
        return {"rel": 8e-3}  # seen: 2e-3
    if case["kind"] == "recurrent":
        return {"rel": 1e-5 if case["cell"] == "lstm" else 2e-3}  # seen: 3e-6, 5e-4
    if case["dtype"] == "bf16":
        return {"rel": 6e-2 if case["activation"] == "relu" else 1e-2}  # seen: 1.5e-2, 2.4e-3
    return {"rel": 5e-3 if case["activation"] == "relu" else 1e-5}  # seen: 1.2e-3, 1e-6


# ------------------------------------------------------------------------------------------------------------------ cases


def listed():
    return [
        # the pixel-vector classifier of the reference's first example, a whole epoch as `Builder.run` drives it: the
        # smallest steps there are, where launches and latency count
        {"name": "mlp_epoch", "kind": "mlp", "call": "epoch", "dtype": "fp32", "inputs": "pixels", "features": 784, "hidden1": 50, "hidden2": 0,
         "hidden3": 0, "classes": 10, "activation": "sigmoid", "batch": 1000, "batches": 10, "rate": 0.01},
        # a tabular classifier in float32 whose sizes divide by nothing
        {"name": "mlp_ragged", "kind": "mlp", "call": "step", "dtype": "fp32", "inputs": "normal", "features": 1003, "hidden1": 770, "hidden2": 330,
         "hidden3": 0, "classes": 17, "activation": "relu", "batch": 700, "rate": 0.001},
        # the wide classifier with bfloat16 products: the largest step
        {"name": "mlp_bf16_wide", "kind": "mlp", "call": "step", "dtype": "bf16", "inputs": "normal", "features": 4096, "hidden1": 4096,
         "hidden2": 4096, "hidden3": 0, "classes": 1000, "activation": "relu", "batch": 8192, "rate": 0.001},
        # the same option at an ordinary size: widths that are multiples of eight but of no tile, ten classes
        {"name": "mlp_bf16_ordinary", "kind": "mlp", "call": "step", "dtype": "bf16", "inputs": "normal", "features": 1000, "hidden1": 1500,
         "hidden2": 600, "hidden3": 0, "classes": 10, "activation": "relu", "batch": 1000, "rate": 0.001},
        # the two-convolution image classifier of the benchmark
        {"name": "cnn_gray", "kind": "cnn", "call": "step", "side": 28, "channels": 1, "filters1": 32, "filters2": 64, "batchnorm": False,
         "pool_stride": 1, "padding": "valid", "hidden": 0, "classes": 10, "batch": 100, "rate": 0.001},
        # the one with batch normalisation, strided pooling and a hidden Dense layer, at its larger batch
        {"name": "cnn_batchnorm", "kind": "cnn", "call": "step", "side": 28, "channels": 1, "filters1": 32, "filters2": 64, "batchnorm": True,
         "pool_stride": 2, "padding": "valid", "hidden": 64, "classes": 10, "batch": 1000, "rate": 0.001},
        # colour images, padded convolutions, filter counts that are multiples of 16 only, an odd batch
        {"name": "cnn_colour", "kind": "cnn", "call": "step", "side": 32, "channels": 3, "filters1": 48, "filters2": 80, "batchnorm": False,
         "pool_stride": 2, "padding": "same", "hidden": 100, "classes": 10, "batch": 125, "rate": 0.001},
        # predictions of the two-convolution classifier for the batch that the estimators evaluate at a time, to the host
        {"name": "cnn_predict", "kind": "cnn", "call": "predict", "side": 28, "channels": 1, "filters1": 32, "filters2": 64, "batchnorm": False,
         "pool_stride": 1, "padding": "valid", "hidden": 0, "classes": 10, "batch": 1000},
        # the sequence regressor of the benchmark
        {"name": "lstm", "kind": "recurrent", "call": "step", "cell": "lstm", "steps": 64, "features": 32, "units1": 256, "units2": 0, "batch": 512,
         "rate": 0.001},
        # two recurrent layers, the first returning its sequence, with ragged sizes everywhere
        {"name": "lstm_stacked", "kind": "recurrent", "call": "step", "cell": "lstm", "steps": 50, "features": 9, "units1": 100, "units2": 60,
         "batch": 130, "rate": 0.001},
        # the optimizer over a flat vector of a large model
        {"name": "adam_flat", "kind": "optimizer", "optimizer": "Adam", "n": 100_000_000},
        # eight partitions' weights and optimizer state averaged after an epoch
        {"name": "average", "kind": "average", "features": 1024, "hidden": 2048, "classes": 1000, "replicas": 8},
    ]


def log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def size(rng, low, high):
    """Half of the sizes people pick are multiples of 8 or more, the others are what the data happens to have."""
    v = log_int(rng, low, high)
    step = rng.choice([1, 1, 8, 32])
    return max(low, v - v % step)


def draw_mlp(rng):
    dtype = rng.choice(["fp32", "bf16"])
    case = {"kind": "mlp", "call": "step", "dtype": dtype, "inputs": rng.choice(["pixels", "normal"]), "features": size(rng, 8, 4096),
            "hidden1": size(rng, 8, 4096), "hidden2": rng.choice([0, size(rng, 8, 4096)]), "hidden3": 0, "classes": size(rng, 2, 1000),
            "activation": rng.choice(["sigmoid", "tanh", "relu"]), "batch": size(rng, 8, 8192), "rate": 0.001}
    if case["hidden2"] and rng.random() < 0.3:
        case["hidden3"] = size(rng, 8, 2048)
    return case, (8e11 if dtype == "bf16" else 6e10)


def draw_cnn(rng, call="step"):
    case = {"kind": "cnn", "call": call, "side": rng.randint(12, 48), "channels": rng.choice([1, 3]), "filters1": size(rng, 8, 64),
            "filters2": size(rng, 8, 128), "batchnorm": rng.random() < 0.4, "pool_stride": rng.choice([1, 2]),
            "padding": rng.choice(["valid", "same"]), "hidden": rng.choice([0, size(rng, 16, 256)]), "classes": size(rng, 2, 100),
            "batch": size(rng, 32, 1000)}
    if call == "step":
        case["rate"] = 0.001
    return case, 3e10


def draw_recurrent(rng):
    units = size(rng, 2, 320)
    return {"kind": "recurrent", "call": "step", "cell": rng.choice(["lstm", "rnn"]), "steps": log_int(rng, 4, 100), "features": size(rng, 1, 64),
            "units1": units, "units2": rng.choice([0, 0, size(rng, 2, 128)]), "batch": size(rng, 8, 512), "rate": 0.001}, 6e10


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "cnn", "cnn", "cnn", "recurrent", "recurrent", "recurrent", "predict", "optimizer", "average"])
    if kind == "optimizer":
        return {"kind": kind, "optimizer": rng.choice(sorted(OPTIMIZERS)), "n": log_int(rng, 10_000, 70_000_000)}
    if kind == "average":
        return {"kind": kind, "features": size(rng, 16, 1024), "hidden": size(rng, 16, 2048), "classes": size(rng, 2, 1000), "replicas": rng.randint(2, 8)}
    if kind == "mlp":
        case, most = draw_mlp(rng)
    elif kind == "recurrent":
        case, most = draw_recurrent(rng)
    else:
        case, most = draw_cnn(rng, "predict" if kind == "predict" else "step")
    least = 32 if kind in ("cnn", "predict") else 8
    while work(case)["flops"] > most and case["batch"] > least:  # a smaller batch where the model is large
        case["batch"] = max(least, case["batch"] // 2)
    return case
