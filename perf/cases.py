"""The work that a program using this package has it do, as cases that can be timed and compared.

A case is a dict of plain values. ``prepare(case, seed)`` lays out what such a program holds before the call (inputs in
device memory, weights, destinations and, for the cases that are issued from a launch recording, the recording),
``run(state)`` makes one pass through the public entry points of ``dali_amd`` and returns every output of it as torch
views of device memory.

Two ways of issuing a pass are in use. "eager" builds and evaluates the expressions anew, as a training loop written
against ``op`` does: host time counts. "recorded" replays a ``Recording`` made once on fixed buffers, as a serving loop
of one shape does: the device's time counts.
"""
import math

import torch

import dali_amd as D
from dali_amd import op

_DTYPES = {"f32": (D.DTYPE_FLOAT, torch.float32, "<f4", 4), "f64": (D.DTYPE_DOUBLE, torch.float64, "<f8", 8), "i32": (D.DTYPE_INT32, torch.int32, "<i4", 4)}
_BY_CODE = {code: (typestr, size) for code, _, typestr, size in _DTYPES.values()}


def listed():
    return [
        # The naive softmax over a batch of scores, the shape that the benchmark's headline is quoted on.
        {"name": "softmax_4096x1024", "kind": "softmax", "issue": "recorded", "outer": 4096, "extent": 1024, "inner": 1},
        # A long elementwise expression, one fused launch over four arrays: the largest arrays the benchmark holds, ...
        {"name": "chain_67108864", "kind": "chain", "issue": "eager", "n": 67108864, "dtype": "f32"},
        # ... and the smallest call: a few thousand values, where building the expression, planning and launching it is all there is.
        {"name": "chain_4001", "kind": "chain", "issue": "eager", "n": 4001, "dtype": "f32"},
        # Reductions of a large matrix along either axis, over everything, and the position of the best entry in each row.
        {"name": "reduce_8192x8192", "kind": "reduce", "issue": "eager", "rows": 8192, "cols": 8192, "dtype": "f32"},
        # The same for statistics kept in double precision over a ragged matrix.
        {"name": "reduce_f64_3001x2047", "kind": "reduce", "issue": "eager", "rows": 3001, "cols": 2047, "dtype": "f64"},
        # Loss and gradient over a large vocabulary ...
        {"name": "xent_8192x32000", "kind": "xent", "issue": "eager", "rows": 8192, "classes": 32000},
        # ... and over a character set: many positions, few and oddly many classes.
        {"name": "xent_51200x97", "kind": "xent", "issue": "recorded", "rows": 51200, "classes": 97},
        # A training step of the output projection of a language model: forward with bias and tanh, then all gradients.
        {"name": "dense_256x1024x32000", "kind": "dense", "issue": "eager", "batch": 256, "inputs": 1024, "outputs": 32000, "dtype": "f32"},
        # One LSTM cell step at a training batch.
        {"name": "lstm_step_256x1024x1024", "kind": "lstm_step", "issue": "recorded", "batch": 256, "inputs": 1024, "hidden": 1024},
        # An LSTM along a sequence at the small batch of a serving loop: a chain of dependent steps.
        {"name": "sequence_lstm_32x8x1024", "kind": "sequence", "issue": "recorded", "cell": "lstm", "steps": 32, "batch": 8, "inputs": 1024, "hidden": 1024},
        # One step of a two-layer LSTM language model: embedding rows, the cells, the projection, the loss with its gradient.
        {"name": "decoder_8x2x1024x32000", "kind": "decoder", "issue": "recorded", "batch": 8, "layers": 2, "hidden": 1024, "vocab": 32000},
        # A training step of a convolution layer: forward, then the gradients of image, filters and bias.
        {"name": "conv_nhwc_32x56x56x64_128x3", "kind": "conv", "issue": "eager", "images": 32, "size": 56, "channels": 64, "filters": 128, "window": 3,
         "stride": 1, "format": "NHWC"},
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], even over its logarithm; a third of them on the round numbers that programs like."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 1 / 3:
        for step in (64, 16, 8):
            if v >= 2 * step:
                v = v // step * step
                break
    return max(low, min(high, v))


def draw(rng):
    kind = rng.choice(["softmax", "chain", "reduce", "xent", "dense", "lstm_step", "sequence", "decoder", "conv"])
    case = {"kind": kind, "issue": rng.choice(["eager", "recorded"])}
    while True:
        if kind == "softmax":
            case.update(outer=_spread(rng, 1, 65536), extent=_spread(rng, 2, 131072), inner=rng.choice([1, 1, 1, _spread(rng, 2, 1024)]))
        elif kind == "chain":
            case.update(n=_spread(rng, 100, 67108864), dtype=rng.choice(["f32", "f32", "f32", "f64"]))
        elif kind == "reduce":
            case.update(rows=_spread(rng, 2, 65536), cols=_spread(rng, 2, 65536), dtype=rng.choice(["f32", "f32", "f64"]))
        elif kind == "xent":
            case.update(rows=_spread(rng, 1, 65536), classes=_spread(rng, 2, 65536))
        elif kind == "dense":
            case.update(batch=_spread(rng, 1, 4096), inputs=_spread(rng, 8, 4096), outputs=_spread(rng, 8, 32000), dtype=rng.choice(["f32", "f32", "f32", "f64"]))
        elif kind == "lstm_step":
            case.update(batch=_spread(rng, 1, 512), inputs=_spread(rng, 16, 2048), hidden=_spread(rng, 16, 2048))
        elif kind == "sequence":
            case.update(cell=rng.choice(["lstm", "gru"]), steps=_spread(rng, 2, 64), batch=_spread(rng, 1, 256), inputs=_spread(rng, 16, 2048), hidden=_spread(rng, 16, 2048))
        elif kind == "decoder":
            case.update(batch=_spread(rng, 1, 128), layers=rng.choice([1, 2, 3]), hidden=_spread(rng, 32, 1536), vocab=_spread(rng, 64, 50257))
        else:
            case.update(images=_spread(rng, 1, 64), size=_spread(rng, 8, 64), channels=_spread(rng, 1, 256), filters=_spread(rng, 8, 256),
                        window=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]), format=rng.choice(["NHWC", "NCHW"]))
        w = work(case)
        if kind in ("softmax", "chain", "xent", "lstm_step") and w["bytes"] < 3.2e7:
            case["issue"] = "eager"  # a single small launch is never worth a recording of its own
        if 2e3 <= w["bytes"] <= 1.0e9 and w["flops"] <= (5e9 if case.get("dtype") == "f64" else 4e10):
            return case


# ------------------------------------------------------------------------------------------------ device memory as tensors
class _View(object):
    """Device memory of an evaluated array for torch: no copy, and the array lives as long as the tensor."""

    def __init__(self, array):
        typestr, size = _BY_CODE[array.dtype]
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": typestr, "data": (array.device_ptr(), False), "version": 2,
                                         "strides": tuple(s * size for s in array.strides) or None}


def _tensor(array):
    return torch.as_tensor(_View(array), device="cuda")


class _Kept(object):
    """A destination that the program keeps from pass to pass."""

    def __init__(self, shape, dtype="f32"):
        self.array = D.Array.empty(shape, _DTYPES[dtype][0])
        self.tensor = _tensor(self.array)

    def assign(self, expression):
        self.array.assign(expression)
        return self


def _outputs(arrays):
    return [a.tensor if isinstance(a, _Kept) else _tensor(a) for a in arrays]


class _Inputs(object):
    """Arrays filled on the device from one seed."""

    def __init__(self, seed):
        torch.cuda.synchronize()
        self._gen = torch.Generator(device="cuda").manual_seed(seed)

    def _make(self, shape, dtype, fill):
        array = D.Array.empty(shape, _DTYPES[dtype][0])
        fill(_tensor(array))
        return array

    def normal(self, shape, dtype="f32", scale=1.0):
        return self._make(shape, dtype, lambda t: t.normal_(0.0, scale, generator=self._gen))

    def uniform(self, shape, low, high, dtype="f32"):
        return self._make(shape, dtype, lambda t: t.uniform_(low, high, generator=self._gen))

    def integers(self, shape, below):
        return self._make(shape, "i32", lambda t: t.random_(0, below, generator=self._gen))

    def glorot(self, rows, cols):
        return self.uniform((rows, cols), -math.sqrt(6.0 / (rows + cols)), math.sqrt(6.0 / (rows + cols)))


# ------------------------------------------------------------------------------------------------ the passes
# Each takes its case and the inputs and returns a function without arguments that makes one pass and returns the
# evaluated arrays. Destinations that a program keeps (activations, gradients) are made here and assigned to.
def _softmax(case, make):
    shape = (case["outer"], case["extent"]) if case["inner"] == 1 else (case["outer"], case["extent"], case["inner"])
    x, out = make.normal(shape), _Kept(shape)
    return lambda: [out.assign(op.softmax(x, 1))]


def _chain(case, make):
    a, b, c, d = (make.uniform((case["n"],), -4.0, 4.0, case["dtype"]) for _ in range(4))
    out = _Kept((case["n"],), case["dtype"])
    return lambda: [out.assign(op.sigmoid(a) * op.tanh(b) + c * d - 0.5 * op.square(a))]


def _reduce(case, make):
    rows, cols, dtype = case["rows"], case["cols"], case["dtype"]
    x = make.normal((rows, cols), dtype)
    columns, lines, best, where = _Kept((cols,), dtype), _Kept((rows,), dtype), _Kept((), dtype), _Kept((rows,), "i32")
    return lambda: [columns.assign(op.sum(x, [0])), lines.assign(op.sum(x, [1])), best.assign(op.max(x)), where.assign(op.argmax(x, 1))]


def _xent(case, make):
    x, t = make.normal((case["rows"], case["classes"]), scale=2.0), make.integers((case["rows"],), case["classes"])
    return lambda: list(op.softmax_cross_entropy(x, t))


def _dense(case, make):
    batch, inputs, outputs, dtype = case["batch"], case["inputs"], case["outputs"], case["dtype"]
    x, dy = make.normal((batch, inputs), dtype), make.normal((batch, outputs), dtype)
    w, b = make.normal((inputs, outputs), dtype, 1.0 / math.sqrt(inputs)), make.normal((1, outputs), dtype, 0.1)
    y, dz, dx, dw, db = (_Kept(s, dtype) for s in ((batch, outputs), (batch, outputs), (batch, inputs), (inputs, outputs), (1, outputs)))

    def step():
        y.assign(op.tanh(op.dot(x, w) + b))
        dz.assign(op.dtanh(y.array) * dy)
        dw.assign(op.dot(x.transpose(), dz.array))
        dx.assign(op.dot(dz.array, w.transpose()))
        db.assign(op.sum(dz.array, [0], True))
        return [y, dw, dx, db]
    return step


def _lstm_step(case, make):
    batch, inputs, hidden = case["batch"], case["inputs"], case["hidden"]
    x, h, c = make.normal((batch, inputs)), make.normal((batch, hidden)), make.normal((batch, hidden))
    w, u, b = make.glorot(inputs, 4 * hidden), make.glorot(hidden, 4 * hidden), make.normal((4 * hidden,), scale=0.1)
    return lambda: list(op.lstm_step(x, h, c, w, u, b))


def _sequence(case, make):
    steps, batch, inputs, hidden = case["steps"], case["batch"], case["inputs"], case["hidden"]
    gates = 4 if case["cell"] == "lstm" else 3
    xs, h, c = make.normal((steps, batch, inputs)), make.normal((batch, hidden)), make.normal((batch, hidden))
    w, u, b = make.glorot(inputs, gates * hidden), make.glorot(hidden, gates * hidden), make.normal((gates * hidden,), scale=0.1)
    if case["cell"] == "lstm":
        return lambda: list(op.lstm_sequence(xs, h, c, w, u, b))
    return lambda: list(op.gru_sequence(xs, h, w, u, b))


def _decoder(case, make):
    batch, layers, hidden, vocab = case["batch"], case["layers"], case["hidden"], case["vocab"]
    table, ids, targets = make.normal((vocab, hidden), scale=0.1), make.integers((batch,), vocab), make.integers((batch,), vocab)
    h, c = ([make.normal((batch, hidden)) for _ in range(layers)] for _ in range(2))
    w, u = ([make.glorot(hidden, 4 * hidden) for _ in range(layers)] for _ in range(2))
    b, out = [make.normal((4 * hidden,), scale=0.1) for _ in range(layers)], make.glorot(hidden, vocab)

    def step():
        c_new, h_new = op.stacked_lstm_step(op.gather(table, ids), h, c, w, u, b)
        logits = op.dot(h_new[-1], out).eval()
        return c_new + h_new + [logits] + list(op.softmax_cross_entropy(logits, targets))
    return step


def _conv(case, make):
    n, size, channels, filters, window, stride, fmt = (case[k] for k in ("images", "size", "channels", "filters", "window", "stride", "format"))
    side = (size - window) // stride + 1
    order = (lambda ch, s: (n, s, s, ch)) if fmt == "NHWC" else (lambda ch, s: (n, ch, s, s))
    x_shape, y_shape = order(channels, size), order(filters, side)
    w_shape = (filters, window, window, channels) if fmt == "NHWC" else (filters, channels, window, window)
    x, w, dy = make.normal(x_shape), make.normal(w_shape, scale=1.0 / math.sqrt(window * window * channels)), make.normal(y_shape)

    def step():
        return [op.conv2d(x, w, stride, stride, "valid", fmt).eval(),
                op.conv2d_backward_input(w, dy, stride, stride, x_shape, "valid", fmt).eval(),
                op.conv2d_backward_filters(x, dy, stride, stride, w_shape, "valid", fmt).eval(),
                op.conv2d_backward_bias(dy, fmt).eval()]
    return step


_KINDS = {"softmax": _softmax, "chain": _chain, "reduce": _reduce, "xent": _xent, "dense": _dense, "lstm_step": _lstm_step, "sequence": _sequence,
          "decoder": _decoder, "conv": _conv}


def prepare(case, seed):
    step = _KINDS[case["kind"]](case, _Inputs(seed))
    torch.cuda.synchronize()  # the inputs were filled on torch's stream; the library has a stream of its own
    if case["issue"] == "eager":
        return {"step": step}
    with D.Recording() as recording:
        outputs = step()
    return {"recording": recording, "outputs": _outputs(outputs)}


def run(state):
    if "recording" in state:
        state["recording"].replay(1)
        return state["outputs"]
    return _outputs(state["step"]())


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind, size = case["kind"], 8 if case.get("dtype") == "f64" else 4
    if kind == "softmax":
        n = case["outer"] * case["extent"] * case["inner"]
        return {"bytes": 2 * 4 * n, "flops": 5 * n}
    if kind == "chain":
        return {"bytes": 5 * size * case["n"], "flops": 8 * case["n"]}
    if kind == "reduce":
        n = case["rows"] * case["cols"]
        return {"bytes": size * (n + case["rows"] + case["cols"] + 1) + 4 * case["rows"], "flops": 4 * n}
    if kind == "xent":
        n = case["rows"] * case["classes"]
        return {"bytes": 4 * (2 * n + 2 * case["rows"] + 1), "flops": 6 * n}
    if kind == "dense":
        batch, inputs, outputs = case["batch"], case["inputs"], case["outputs"]
        return {"bytes": size * (2 * batch * inputs + 2 * inputs * outputs + 2 * batch * outputs + 2 * outputs), "flops": 6 * batch * inputs * outputs}
    if kind in ("lstm_step", "sequence"):
        batch, inputs, hidden, steps, gates = case["batch"], case["inputs"], case["hidden"], case.get("steps", 1), 3 if case.get("cell") == "gru" else 4
        values = gates * hidden * (inputs + hidden + 1) + batch * (steps * (inputs + hidden) + 3 * hidden)
        return {"bytes": 4 * values, "flops": 2 * steps * batch * (inputs + hidden) * gates * hidden}
    if kind == "decoder":
        batch, layers, hidden, vocab = case["batch"], case["layers"], case["hidden"], case["vocab"]
        values = layers * (4 * hidden * (2 * hidden + 1) + 4 * batch * hidden) + hidden * vocab + 2 * batch * vocab + 2 * batch * hidden
        return {"bytes": 4 * values, "flops": 2 * batch * hidden * (8 * layers * hidden + vocab)}
    n, channels, filters, window = case["images"], case["channels"], case["filters"], case["window"]
    side = (case["size"] - window) // case["stride"] + 1
    values = 2 * n * case["size"] ** 2 * channels + 2 * n * side ** 2 * filters + 2 * window ** 2 * channels * filters + filters
    return {"bytes": 4 * values, "flops": 6 * n * side ** 2 * filters * window ** 2 * channels}


# About four times the distance from the same pass in double precision (largest over these cases and two dozen drawn ones):
# elementwise maps and softmax 1.0e-7, sums 2.9e-7, products and the recurrences built on them 1.2e-6, in double precision 4.3e-16.
_TOLERANCES = {"softmax": (5e-7, 3e-6), "chain": (2e-7, 1.5e-6), "reduce": (1.2e-6, 6e-6), "xent": (5e-7, 3e-6), "dense": (5e-6, 3e-5), "lstm_step": (2e-6, 3e-5),
               "sequence": (2e-6, 3e-5), "decoder": (2e-6, 1e-5), "conv": (5e-6, 3e-5)}


def tolerance(case):
    rel, most = (2e-15, 2e-14) if case.get("dtype") == "f64" else _TOLERANCES[case["kind"]]
    return {"rel": rel, "max": most}
