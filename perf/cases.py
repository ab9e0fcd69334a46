"""What is measured when this library's speed is in question: passes of the work that a program built on the tensor
API has it do, from a bias row added to a batch of 128 digits to an optimizer step over 2^28 parameters.

A case is a dict of plain values.  ``prepare`` makes what such a program has in hand before the call (tensors in
device memory, layers, optimizer state), ``run`` is one pass through the public entry points: the tensor API, the
layers and the optimizers.  Device memory comes from torch, so that the outputs of a pass can be handed back as
tensors; the library works on the same pointers.  Sizes are those of the benchmark and of the tests of this
repository, or generic.
"""
from __future__ import annotations

import math

import torch

from cortex_amd import dimensions as dims
from cortex_amd import driver as drv
from cortex_amd import nn_layers as layers
from cortex_amd import optimize
from cortex_amd import tensor as ct

_TORCH = {"float": torch.float32, "double": torch.float64, "int": torch.int32, "ubyte": torch.uint8}
_NAME = {v: k for k, v in _TORCH.items()}
_SIZE = {"float": 4, "double": 8, "int": 4, "ubyte": 1}


# ------------------------------------------------------------------------------------------------- the cases

def listed() -> list:
    return [
        # The bias of a small linear layer over one batch of digits (28 x 28): the smallest call that layers make, where
        # latency is everything.
        {"name": "bias_add_small", "kind": "bias", "rows": 128, "columns": 784, "op": "+", "datatype": "float"},
        # A batch of byte images on its way into a network: converted, the channel means taken off, scaled.
        {"name": "normalize_images", "kind": "images", "batch": 256, "channels": 3, "side": 224, "interleaved": False},
        # An activation over a transposed view, written contiguous: the strided elementwise path.
        {"name": "transposed_tanh", "kind": "transposed", "rows": 8192, "columns": 8192, "op": "tanh", "datatype": "float"},
        # Sums over the rows and over the columns (a transposed view) of one matrix: statistics, norms, losses.
        {"name": "reduce_float", "kind": "reduce", "rows": 16384, "columns": 4096, "op": "sum", "datatype": "float"},
        {"name": "reduce_double", "kind": "reduce", "rows": 4096, "columns": 4096, "op": "magnitude-squared",
         "datatype": "double"},
        # The optimizer step over all the parameters of a large network.
        {"name": "adam_large", "kind": "optimizer", "optimizer": "adam", "parameters": 1 << 28, "datatype": "float"},
        # A training step of a small network on digits (784 -> 128 -> 10, dropout between): forward, loss gradient,
        # backward and optimizer, some twenty-five small calls in a row.
        {"name": "mlp_training_step", "kind": "mlp", "batch": 128, "inputs": 784, "hidden": 128, "classes": 10,
         "activation": "relu", "datatype": "float"},
        # A wide linear layer, forward and backward: three matrix products.
        {"name": "linear_wide", "kind": "linear", "batch": 1024, "inputs": 4096, "outputs": 4096, "datatype": "float"},
        # Convolutional layers, forward and backward: one of an image network and a small one of a digit network.
        {"name": "convolution_images", "kind": "convolution", "batch": 64, "channels": 64, "kernels": 64, "side": 56,
         "window": 3, "pad": 1, "stride": 1, "datatype": "float"},
        {"name": "convolution_digits", "kind": "convolution", "batch": 128, "channels": 16, "kernels": 32, "side": 28,
         "window": 3, "pad": 1, "stride": 1, "datatype": "float"},
        # What stands between two convolutions, in training: normalization, activation and pooling, forward and backward.
        {"name": "normalize_activate_pool", "kind": "block", "norm": "batch", "batch": 32, "channels": 64, "side": 112,
         "window": 3, "pad": 1, "stride": 2, "activation": "relu", "datatype": "float"},
        # Class centers kept beside a network: rows looked up by label, the differences added back by label.
        {"name": "label_rows", "kind": "labels", "batch": 65536, "classes": 32768, "width": 1024, "datatype": "float"},
    ]


def _log_int(rng, low: int, high: int) -> int:
    """A whole number in [low, high], even over its logarithm; powers of two are no likelier than others."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_bias(rng):
    while True:
        case = {"rows": _log_int(rng, 1, 16384), "columns": _log_int(rng, 1, 16384)}
        if case["rows"] * case["columns"] >= 64:
            break
    return dict(case, op=rng.choice(["+", "+", "*", "max"]), datatype=rng.choice(["float", "float", "double", "int"]))


def _draw_images(rng):
    return {"batch": _log_int(rng, 1, 256), "channels": rng.choice([1, 3, 3, 4]), "side": _log_int(rng, 28, 256),
            "interleaved": rng.random() < 0.5}


def _draw_transposed(rng):
    return {"rows": _log_int(rng, 64, 8192), "columns": _log_int(rng, 64, 8192),
            "op": rng.choice(["exp", "tanh", "logistic", "sqrt"]), "datatype": rng.choice(["float", "float", "double"])}


def _draw_reduce(rng):
    return {"rows": _log_int(rng, 10, 16384), "columns": _log_int(rng, 10, 8192),
            "op": rng.choice(["sum", "mean", "max", "magnitude-squared", "magnitude"]),
            "datatype": rng.choice(["float", "float", "double", "int"])}


def _draw_optimizer(rng):
    return {"optimizer": rng.choice(["adam", "adam", "adadelta", "sgd"]), "parameters": _log_int(rng, 1000, 1 << 26),
            "datatype": rng.choice(["float", "float", "double"])}


def _draw_mlp(rng):
    return {"batch": _log_int(rng, 1, 2048), "inputs": _log_int(rng, 64, 4096), "hidden": _log_int(rng, 16, 2048),
            "classes": _log_int(rng, 2, 1000), "activation": rng.choice(["relu", "tanh", "logistic"]),
            "datatype": rng.choice(["float", "float", "float", "double"])}


def _draw_linear(rng):
    return {"batch": _log_int(rng, 16, 4096), "inputs": _log_int(rng, 16, 4096), "outputs": _log_int(rng, 10, 4096),
            "datatype": rng.choice(["float", "float", "float", "double"])}


def _draw_convolution(rng):
    while True:
        window, stride = rng.choice([1, 3, 3, 3, 5]), rng.choice([1, 1, 1, 2])
        case = {"batch": _log_int(rng, 1, 256), "channels": _log_int(rng, 1, 256), "kernels": _log_int(rng, 4, 256),
                "side": _log_int(rng, 7, 112), "window": window, "pad": rng.choice([0, window // 2]), "stride": stride,
                "datatype": rng.choice(["float", "float", "float", "float", "double"])}
        cells = case["batch"] * case["channels"] * window ** 2 * _conv_side(case) ** 2
        if cells <= 1 << 28 and cells * case["kernels"] <= 1 << 34:
            return case


def _draw_block(rng):
    while True:
        window = rng.choice([2, 3])
        case = {"norm": rng.choice(["batch", "batch", "local"]), "batch": _log_int(rng, 1, 128),
                "channels": _log_int(rng, 4, 256), "side": _log_int(rng, 7, 112), "window": window,
                "pad": rng.choice([0, window // 2]), "stride": 2, "activation": rng.choice(["relu", "relu", "tanh"]),
                "datatype": rng.choice(["float", "float", "float", "double"])}
        if case["batch"] * case["channels"] * case["side"] ** 2 <= 1 << 25:
            return case


def _draw_labels(rng):
    while True:
        case = {"batch": _log_int(rng, 64, 65536), "classes": _log_int(rng, 10, 32768), "width": _log_int(rng, 10, 1024)}
        # entries that fall on one row are added one after the other, in their order: no class holds more than a share
        if case["batch"] <= 64 * case["classes"]:
            return dict(case, datatype=rng.choice(["float", "float", "double"]))


_DRAW = {"bias": _draw_bias, "images": _draw_images, "transposed": _draw_transposed, "reduce": _draw_reduce,
         "optimizer": _draw_optimizer, "mlp": _draw_mlp, "linear": _draw_linear, "convolution": _draw_convolution,
         "block": _draw_block, "labels": _draw_labels}


def draw(rng) -> dict:
    kind = rng.choice(sorted(_DRAW))
    return dict(_DRAW[kind](rng), kind=kind)


# ------------------------------------------------------------------------------------------------- shared pieces

class _State:
    """What a pass works on.  Buffers that layers allocate from the library are given back with the state."""

    def __init__(self, case: dict, seed: int):
        self.case = case
        self.datatype = case.get("datatype", "float")
        self.generator = torch.Generator(device="cuda").manual_seed(seed)
        self.device = _device()
        self.stream = drv.HipStream(self.device, torch.cuda.current_stream().cuda_stream or None)
        self.stream.seed_random(seed)
        self.owned = []
        self.outputs = []

    def __del__(self):
        for buffer in self.owned:
            buffer.release()

    def uniform(self, *shape, low=0.0, high=1.0, dtype=None):
        return torch.empty(shape, device="cuda", dtype=dtype or _TORCH[self.datatype]).uniform_(
            low, high, generator=self.generator)

    def normal(self, *shape, mean=0.0, std=1.0, dtype=None):
        return torch.empty(shape, device="cuda", dtype=dtype or _TORCH[self.datatype]).normal_(
            mean, std, generator=self.generator)

    def integers(self, *shape, low, high, dtype):
        return torch.randint(low, high, shape, device="cuda", dtype=dtype, generator=self.generator)

    def zeros(self, *shape, dtype=None):
        return torch.zeros(shape, device="cuda", dtype=dtype or _TORCH[self.datatype])

    def tensor(self, t: torch.Tensor) -> ct.Tensor:
        """The library's view of a torch tensor; the tensor lives as long as the view."""
        buffer = drv.DeviceBuffer(self.device, t.data_ptr(), t.numel(), _NAME[t.dtype])
        buffer.storage = t
        return ct.Tensor(self.device, dims.dimensions(list(t.shape)), buffer)

    def output(self, t: torch.Tensor) -> ct.Tensor:
        self.outputs.append(t)
        return self.tensor(t)

    def layer(self, description: dict, batch: int):
        layer = layers.create(description, batch, self.datatype)
        for value in vars(layer).values():
            if ct.is_tensor(value) and value.buffer not in self.owned:
                self.owned.append(value.buffer)
        return layer


_DEVICE = None


def _device():
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = drv.HipDriver().default_device()
    return _DEVICE


def _conv_side(case: dict) -> int:
    return (case["side"] + 2 * case["pad"] - case["window"]) // case["stride"] + 1


def _pool_side(case: dict) -> int:
    return -(-(case["side"] + 2 * case["pad"] - case["window"]) // case["stride"]) + 1


# ------------------------------------------------------------------------------------------------- bias

def _prepare_bias(s: _State):
    r, c = s.case["rows"], s.case["columns"]
    if s.datatype == "int":
        x, y = (s.integers(*shape, low=-1000, high=1000, dtype=torch.int32) for shape in ((r, c), (c,)))
    else:
        x, y = s.uniform(r, c, low=-1.0), s.uniform(c, low=-1.0)
    s.x, s.y = s.tensor(x), s.tensor(y)
    s.dest = s.output(s.zeros(r, c))


def _run_bias(s: _State):
    ct.binary_op(s.dest, 1.0, s.x, 1.0, s.y, s.case["op"])


def _work_bias(c):
    n = c["rows"] * c["columns"]
    return (2 * n + c["columns"]) * _SIZE[c["datatype"]], n


# ------------------------------------------------------------------------------------------------- images

def _prepare_images(s: _State):
    n, c, side = s.case["batch"], s.case["channels"], s.case["side"]
    shape = (n, side, side, c) if s.case["interleaved"] else (n, c, side, side)
    pixels = s.tensor(s.integers(*shape, low=0, high=256, dtype=torch.uint8))
    s.pixels = ct.transpose(pixels, [0, 3, 1, 2]) if s.case["interleaved"] else pixels
    s.mean = ct.in_place_reshape(s.tensor(s.uniform(c, low=100.0, high=130.0)), [c, 1, 1])
    s.deviation = ct.in_place_reshape(s.tensor(s.uniform(c, low=50.0, high=70.0)), [c, 1, 1])
    s.converted = s.output(s.zeros(n, c, side, side))
    s.centered = s.output(s.zeros(n, c, side, side))
    s.normalized = s.output(s.zeros(n, c, side, side))


def _run_images(s: _State):
    ct.assign(s.converted, s.pixels)
    ct.binary_op(s.centered, 1.0, s.converted, 1.0, s.mean, "-")
    ct.binary_op(s.normalized, 1.0, s.centered, 1.0, s.deviation, "/")


def _work_images(c):
    n = c["batch"] * c["channels"] * c["side"] ** 2
    return n + 5 * 4 * n, 2 * n


# ------------------------------------------------------------------------------------------------- transposed

def _prepare_transposed(s: _State):
    r, c = s.case["rows"], s.case["columns"]
    x = s.normal(c, r)
    if s.case["op"] == "sqrt":
        x.abs_()
    s.x = ct.transpose(s.tensor(x), [1, 0])
    s.dest = s.output(s.zeros(r, c))


def _run_transposed(s: _State):
    ct.unary_op(s.dest, 1.0, s.x, s.case["op"])


def _work_transposed(c):
    n = c["rows"] * c["columns"]
    return 2 * n * _SIZE[c["datatype"]], n


# ------------------------------------------------------------------------------------------------- reduce

def _prepare_reduce(s: _State):
    r, c = s.case["rows"], s.case["columns"]
    x = s.integers(r, c, low=-100, high=100, dtype=torch.int32) if s.datatype == "int" else s.normal(r, c)
    s.x = s.tensor(x)
    s.x_t = ct.transpose(s.x, [1, 0])
    s.of_rows = s.output(s.zeros(r, 1))
    s.of_columns = s.output(s.zeros(c, 1))


def _run_reduce(s: _State):
    ct.unary_reduce(s.of_rows, 1.0, s.x, s.case["op"])
    ct.unary_reduce(s.of_columns, 1.0, s.x_t, s.case["op"])


def _work_reduce(c):
    n = c["rows"] * c["columns"]
    return (2 * n + c["rows"] + c["columns"]) * _SIZE[c["datatype"]], 2 * n


# ------------------------------------------------------------------------------------------------- optimizer

def _prepare_optimizer(s: _State):
    n = s.case["parameters"]
    s.parameters = s.output(s.uniform(n, low=-0.05, high=0.05))
    s.gradient = s.tensor(s.normal(n, std=1e-3))
    kind = s.case["optimizer"]
    # the state of a run that has been going for a while
    if kind == "adam":
        s.memory = {"m": s.output(s.normal(n, std=1e-4)), "v": s.output(s.uniform(n, low=5e-7, high=2e-6))}
        description = optimize.adam()
    elif kind == "adadelta":
        s.memory = {"grad-accum": s.output(s.uniform(n, low=5e-7, high=2e-6)),
                    "dx-accum": s.output(s.uniform(n, low=5e-9, high=2e-8))}
        description = optimize.adadelta()
    else:
        s.memory = {"momentum-vals": s.output(s.normal(n, std=1e-5))}
        description = optimize.sgd()
    s.optimizer = optimize.create_optimizer(optimize.Backend(s.stream, s.datatype), description)
    if kind == "sgd":
        s.optimizer._temp = ct.new_tensor([n], s.datatype, init_value=None)
        s.owned.append(s.optimizer._temp.buffer)
    for _ in range(10):
        s.optimizer = s.optimizer.batch_update()


def _run_optimizer(s: _State):
    s.optimizer = s.optimizer.batch_update()
    s.optimizer.compute_parameters(s.memory, 1.0, 0, s.gradient, s.parameters)


def _work_optimizer(c):
    n, size = c["parameters"], _SIZE[c["datatype"]]
    reads_writes, flops = {"adam": (7, 15), "adadelta": (7, 15), "sgd": (5, 6)}[c["optimizer"]]
    return reads_writes * n * size, flops * n


# ------------------------------------------------------------------------------------------------- layers

def _entry(s: _State, buffer: torch.Tensor, gradient: torch.Tensor = None, returned=True) -> dict:
    """A buffer and its gradient as the layers take them; both are outputs of the pass unless said otherwise."""
    keep = s.output if returned else s.tensor
    return {"buffer": keep(buffer), "gradient": keep(torch.zeros_like(buffer) if gradient is None else gradient)}


def _linear_parameters(s: _State, n_in: int, n_out: int) -> dict:
    return {"weights": _entry(s, s.normal(n_out, n_in, std=math.sqrt(2.0 / n_in))),
            "bias": _entry(s, s.uniform(n_out, low=-0.05, high=0.05))}


def _clear_gradients(parameters: dict) -> None:
    for entry in parameters.values():
        ct.assign(entry["gradient"], 0)


def _prepare_mlp(s: _State):
    b, n_in, hidden, classes = (s.case[k] for k in ("batch", "inputs", "hidden", "classes"))
    s.input = {"buffer": s.tensor(s.uniform(b, n_in)), "gradient": None}
    labels = s.zeros(b, classes)
    labels[torch.arange(b, device="cuda"), s.integers(b, low=0, high=classes, dtype=torch.int64)] = 1.0
    s.labels = {"buffer": s.tensor(labels)}
    s.parameters = [_linear_parameters(s, n_in, hidden), _linear_parameters(s, hidden, classes)]
    s.edges = [s.input] + [_entry(s, s.zeros(b, n)) for n in (hidden, hidden, hidden, classes, classes)]
    s.layers = [s.layer(description, b) for description in (
        {"type": "linear"}, {"type": s.case["activation"]},
        {"type": "dropout", "distribution": "bernoulli", "probability": 0.8, "input-size": hidden},
        {"type": "linear"}, {"type": "softmax"})]
    s.of_layer = {0: s.parameters[0], 3: s.parameters[1]}
    buffers = [entry for p in s.parameters for entry in p.values()]
    total = sum(e["buffer"].ecount() for e in buffers)
    s.memory = {"m": s.output(s.normal(total, std=1e-4)), "v": s.output(s.uniform(total, low=5e-7, high=2e-6))}
    s.optimizer = optimize.create_optimizer(optimize.Backend(s.stream, s.datatype), optimize.adam())
    for _ in range(10):
        s.optimizer = s.optimizer.batch_update()


def _run_mlp(s: _State):
    for p in s.parameters:
        _clear_gradients(p)
    for i, layer in enumerate(s.layers):
        if hasattr(layer, "prepare_forward"):
            layer.prepare_forward(s.of_layer.get(i, {}), [s.edges[i]], [s.edges[i + 1]])
        layer.forward(s.of_layer.get(i, {}), [s.edges[i]], [s.edges[i + 1]])
    layers.softmax_loss_gradient({"output": s.edges[-1], "labels": s.labels})
    for i in reversed(range(len(s.layers))):
        s.layers[i].backward(s.of_layer.get(i, {}), [s.edges[i + 1]], [s.edges[i]])
    s.optimizer = s.optimizer.batch_update()
    offset = 0
    for p in s.parameters:
        for entry in p.values():
            s.optimizer.compute_parameters(s.memory, 1.0 / s.case["batch"], offset, entry["gradient"], entry["buffer"])
            offset += entry["buffer"].ecount()


def _work_mlp(c):
    b, n_in, hidden, classes = (c[k] for k in ("batch", "inputs", "hidden", "classes"))
    parameters = (n_in + 1) * hidden + (hidden + 1) * classes
    values = b * (n_in + 6 * hidden + 5 * classes) + 8 * parameters
    flops = 4 * b * n_in * hidden + 6 * b * hidden * classes + 20 * b * hidden + 15 * parameters
    return values * _SIZE[c["datatype"]], flops


def _prepare_linear(s: _State):
    b, n_in, n_out = (s.case[k] for k in ("batch", "inputs", "outputs"))
    s.layers = [s.layer({"type": "linear"}, b)]
    s.parameters = _linear_parameters(s, n_in, n_out)
    s.inputs = [_entry(s, s.uniform(b, n_in))]
    s.results = [_entry(s, s.zeros(b, n_out), s.normal(b, n_out, std=1e-3))]


def _run_layers_with_parameters(s: _State):
    _clear_gradients(s.parameters)
    s.layers[0].forward(s.parameters, s.inputs, s.results)
    s.layers[0].backward(s.parameters, s.results, s.inputs)


def _work_linear(c):
    b, n_in, n_out = (c[k] for k in ("batch", "inputs", "outputs"))
    values = 2 * b * n_in + 2 * b * n_out + 2 * n_in * n_out + 2 * n_out
    return values * _SIZE[c["datatype"]], 6 * b * n_in * n_out


def _prepare_convolution(s: _State):
    b, cin, cout, side, k = (s.case[n] for n in ("batch", "channels", "kernels", "side", "window"))
    description = layers.convolutional(k, s.case["pad"], s.case["stride"], cout,
                                       {"channels": cin, "height": side, "width": side})
    out = description["output-dimension"]["height"]
    s.layers = [s.layer(description, b)]
    s.parameters = _linear_parameters(s, cin * k * k, cout)
    s.inputs = [_entry(s, s.normal(b, cin, side, side).clamp_(min=0.0))]
    s.results = [_entry(s, s.zeros(b, cout, out, out), s.normal(b, cout, out, out, std=1e-3))]


def _work_convolution(c):
    size, side = c["side"] ** 2, _conv_side(c) ** 2
    weights = c["kernels"] * c["channels"] * c["window"] ** 2
    values = c["batch"] * (2 * c["channels"] * size + 2 * c["kernels"] * side) + 2 * weights + 2 * c["kernels"]
    return values * _SIZE[c["datatype"]], 6 * c["batch"] * weights * side


def _prepare_block(s: _State):
    b, c, side, k = (s.case[n] for n in ("batch", "channels", "side", "window"))
    dimension = {"channels": c, "height": side, "width": side}
    pool = layers.max_pooling(k, s.case["pad"], s.case["stride"], dimension)
    out = pool["output-dimension"]["height"]
    if s.case["norm"] == "batch":
        norm = {"type": "batch-normalization", "mode": "spatial", "epsilon": 1e-4, "average-factor": 0.9,
                "input-dimension": dimension}
        s.parameters = {"scale": _entry(s, s.uniform(c, low=0.5, high=1.5)), "bias": _entry(s, s.normal(c, std=0.1)),
                        "means": {"buffer": s.output(s.zeros(c))}, "variances": {"buffer": s.output(s.zeros(c))}}
    else:
        norm = layers.local_response_normalization(dimension)
        s.parameters = {}
    s.layers = [s.layer(d, b) for d in (norm, {"type": s.case["activation"]}, pool)]
    s.edges = [_entry(s, s.normal(b, c, side, side, mean=0.2)), _entry(s, s.zeros(b, c, side, side)),
               _entry(s, s.zeros(b, c, side, side)),
               _entry(s, s.zeros(b, c, out, out), s.normal(b, c, out, out, std=1e-3))]


def _run_block(s: _State):
    for i, layer in enumerate(s.layers):
        layer.forward(s.parameters if i == 0 else {}, [s.edges[i]], [s.edges[i + 1]])
    # pooling adds onto the gradient that it propagates
    ct.assign(s.edges[2]["gradient"], 0)
    for i in reversed(range(len(s.layers))):
        s.layers[i].backward(s.parameters if i == 0 else {}, [s.edges[i + 1]], [s.edges[i]])


def _work_block(c):
    n, m = (c["batch"] * c["channels"] * side ** 2 for side in (c["side"], _pool_side(c)))
    # normalization 2 + 3 or 4, activation 2 + 3, clearing 1, pooling 1 and 3 of the large tensors; 1 + 2 of the pooled one
    values = (15 if c["norm"] == "batch" else 16) * n + 3 * m
    return values * _SIZE[c["datatype"]], 25 * n + 2 * c["window"] ** 2 * m


# ------------------------------------------------------------------------------------------------- labels

def _prepare_labels(s: _State):
    b, classes, width = (s.case[k] for k in ("batch", "classes", "width"))
    s.features = s.tensor(s.normal(b, width))
    s.indexes = s.tensor(s.integers(b, low=0, high=classes, dtype=torch.int32))
    s.centers = s.output(s.normal(classes, width))
    s.looked_up = s.output(s.zeros(b, width))
    s.differences = s.output(s.zeros(b, width))


def _run_labels(s: _State):
    chosen = ct.select(s.centers, s.indexes, "all")
    ct.assign(s.looked_up, chosen)
    ct.binary_op(s.differences, 1.0, s.features, 1.0, s.looked_up, "-")
    ct.binary_op(chosen, 1.0, chosen, 1e-3, s.differences, "+")


def _work_labels(c):
    b, width = c["batch"], c["width"]
    touched = c["classes"] * (1.0 - math.exp(-b / c["classes"]))   # rows that at least one label selects
    values = touched * width * 3 + b * width * 5
    return int(values * _SIZE[c["datatype"]] + 8 * b), 3 * b * width


# ------------------------------------------------------------------------------------------------- the interface

_KINDS = {
    "bias": (_prepare_bias, _run_bias, _work_bias),
    "images": (_prepare_images, _run_images, _work_images),
    "transposed": (_prepare_transposed, _run_transposed, _work_transposed),
    "reduce": (_prepare_reduce, _run_reduce, _work_reduce),
    "optimizer": (_prepare_optimizer, _run_optimizer, _work_optimizer),
    "mlp": (_prepare_mlp, _run_mlp, _work_mlp),
    "linear": (_prepare_linear, _run_layers_with_parameters, _work_linear),
    "convolution": (_prepare_convolution, _run_layers_with_parameters, _work_convolution),
    "block": (_prepare_block, _run_block, _work_block),
    "labels": (_prepare_labels, _run_labels, _work_labels),
}


def prepare(case: dict, seed: int):
    state = _State(case, seed)
    with ct.tensor_context(state.stream, state.datatype):
        _KINDS[case["kind"]][0](state)
    return state


def run(state):
    with ct.tensor_context(state.stream, state.datatype):
        _KINDS[state.case["kind"]][1](state)
    return state.outputs


def work(case: dict) -> dict:
    nbytes, flops = _KINDS[case["kind"]][2](case)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    """About four times what the float passes differ by from the same passes in double precision."""
    kind, double = case["kind"], case.get("datatype") == "double"
    if kind in ("bias", "images", "labels", "optimizer"):
        return "exact"       # one rounding per stored value, in a fixed order
    if kind == "reduce":
        # exact whatever the order: maxima, and sums of whole numbers; the others are sums in double rounded once
        if case["op"] == "max" or case["datatype"] == "int":
            return "exact"
        return {"rel": 1e-14 if double else 1e-7}
    if kind == "transposed":
        if case["op"] == "sqrt":
            return "exact"
        return {"rel": 1e-14 if double else 2e-7}
    if double:
        return {"rel": 1e-13}
    # A value within a rounding error of zero under relu, or of another value of its pooling window, moves a whole
    # gradient to the other side: 7e-4 seen over a few million values.
    if kind == "block" or (kind == "mlp" and case["activation"] == "relu"):
        return {"rel": 3e-3}
    # sums of products in the tensors' own precision, over up to a few thousand terms: 1e-6 seen
    return {"rel": 4e-6}


# ------------------------------------------------------------------------------------------------- in 64 bits

def _storage(t: ct.Tensor) -> torch.Tensor:
    return t.buffer.storage.double()


def _exact_transposed(s: _State):
    x = _storage(s.x).t()
    return [{"exp": torch.exp, "tanh": torch.tanh, "logistic": torch.sigmoid, "sqrt": torch.sqrt}[s.case["op"]](x)]


def _exact_reduce(s: _State):
    x = _storage(s.x)
    of = {"sum": torch.sum, "mean": torch.mean, "max": torch.amax,
          "magnitude-squared": lambda v, dim, keepdim: (v * v).sum(dim, keepdim=keepdim),
          "magnitude": lambda v, dim, keepdim: (v * v).sum(dim, keepdim=keepdim).sqrt()}[s.case["op"]]
    return [of(x, dim=1, keepdim=True), of(x, dim=0, keepdim=True).t()]


def _exact_linear(s: _State):
    weights, bias = (_storage(s.parameters[k]["buffer"]) for k in ("weights", "bias"))
    x, gradient = _storage(s.inputs[0]["buffer"]), _storage(s.results[0]["gradient"])
    return [weights, gradient.t() @ x, bias, gradient.sum(0), x, gradient @ weights, x @ weights.t() + bias, gradient]


def _exact_convolution(s: _State):
    weights, bias = (_storage(s.parameters[k]["buffer"]) for k in ("weights", "bias"))
    x, gradient = _storage(s.inputs[0]["buffer"]), _storage(s.results[0]["gradient"])
    window = {"kernel_size": s.case["window"], "padding": s.case["pad"], "stride": s.case["stride"]}
    result, x_gradient = torch.empty_like(gradient), torch.empty_like(x)
    weight_gradient = torch.zeros_like(weights)
    for image in range(len(x)):
        cells, g = torch.nn.functional.unfold(x[image:image + 1], **window)[0], gradient[image].flatten(1)
        result[image] = (weights @ cells + bias[:, None]).view_as(result[image])
        weight_gradient += g @ cells.t()
        x_gradient[image] = torch.nn.functional.fold((weights.t() @ g)[None], x.shape[2:], **window)[0]
    return [weights, weight_gradient, bias, gradient.sum((0, 2, 3)), x, x_gradient, result, gradient]


def _exact_block(s: _State):
    if s.case["norm"] != "batch":
        return None
    # The gradients have no such value where rounding decides which element of a window is the largest.
    scale, bias = (_storage(s.parameters[k]["buffer"])[:, None, None] for k in ("scale", "bias"))
    x = _storage(s.edges[0]["buffer"])
    variance, mean = torch.var_mean(x, dim=(0, 2, 3), keepdim=True, correction=0)
    normalized = scale * (x - mean) / torch.sqrt(variance + 1e-4) + bias
    active = torch.clamp(normalized, min=0.0) if s.case["activation"] == "relu" else torch.tanh(normalized)
    return [scale.flatten(), None, bias.flatten(), None, None, None, x, None, normalized, None, active, None, None, None]


_EXACT = {"transposed": _exact_transposed, "reduce": _exact_reduce, "linear": _exact_linear,
          "convolution": _exact_convolution, "block": _exact_block}


def exact(case: dict, seed: int):
    """None where a pass rounds once per stored value, in a fixed order, and is compared to the bit, and for the whole
    training step, whose dropout mask only the library's generator gives."""
    if case["kind"] not in _EXACT or case.get("datatype") == "int":
        return None
    return _EXACT[case["kind"]](prepare(case, seed))
