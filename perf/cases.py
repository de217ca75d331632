"""What a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values; its ``"kind"`` names the path it takes through the public entry points:

``conv``       one convolution layer, forward and backward (dX, dW, db): ``nn.functional.conv2d`` and ``Tensor.backward``
``pool``       one max-pool, forward and backward: ``nn.functional.max_pool2d`` and ``Tensor.backward``
``small_net``  the README network, one training step (forward, backward, SGD); ``"graph"``: the step is recorded once
               with ``StepGraph`` and replayed
``train``      ResNet-18, one training step, batch-statistics normalisation, everything resident on the device
``infer``      ResNet-18, forward only, moving statistics, in float32 or with bf16 convolutions

Everything is float32 at the interface; ``"precision": "bf16"`` is the package's opt-in ``conv_precision('bf16')``.
Outputs are handed over as torch views of the package's own device arrays: nothing is copied.
"""
import math

import numpy as np
import torch

import xshinnosuke_amd as xs
from xshinnosuke_amd import backend as be
from xshinnosuke_amd.layers import (AvgPooling2D, BatchNormalization, Conv2D, Dense, Flatten, MaxPooling2D, ReLU)
from xshinnosuke_amd.nn import functional as F
from xshinnosuke_amd.nn.models import Module, Sequential
from xshinnosuke_amd.optim import SGD


# --------------------------------------------------------------------------- the cases
def listed():
    return [
        # The README network at its own size: eleven million multiplications, a dozen launches, bound by the host.
        {"name": "small_net_n256", "kind": "small_net", "n": 256, "size": 28, "filters": 8, "graph": False},
        # The same step recorded and replayed, what fit() does under GLOBAL.STEP_GRAPH: launch latency on the device.
        {"name": "small_net_graph_n256", "kind": "small_net", "n": 256, "size": 28, "filters": 8, "graph": True},
        # The benchmark's convolution: a layer of ResNet-18's first stage at the training batch.
        {"name": "conv_64_56_n32", "kind": "conv", "n": 32, "c": 64, "h": 56, "w": 56, "k": 64, "r": 3, "stride": 1, "pad": 1,
         "relu": False, "precision": "fp32"},
        # A stage's first convolution: more filters, half the resolution.
        {"name": "conv_128_256_s2_n32", "kind": "conv", "n": 32, "c": 128, "h": 28, "w": 28, "k": 256, "r": 3, "stride": 2,
         "pad": 1, "relu": False, "precision": "fp32"},
        # No size is a round one: images of another camera, 5x5 filters, a bias and a ReLU in the layer itself.
        {"name": "conv_ragged_5x5_n7", "kind": "conv", "n": 7, "c": 24, "h": 45, "w": 61, "k": 40, "r": 5, "stride": 1, "pad": 2,
         "relu": True, "precision": "fp32"},
        # Training of a layer with the bf16 opt-in (the weight gradient stays in float32).
        {"name": "conv_bf16_128_28_n32", "kind": "conv", "n": 32, "c": 128, "h": 28, "w": 28, "k": 128, "r": 3, "stride": 1,
         "pad": 1, "relu": False, "precision": "bf16"},
        # The benchmark's max-pool: behind the first convolution of ResNet-18, 5 % ties.
        {"name": "pool_64_112_n32", "kind": "pool", "n": 32, "c": 64, "h": 112, "w": 112, "k": 3, "stride": 2, "pad": 1},
        # The reference's own timing script: 56x56 images, 100 classes, here at a batch of 32.
        {"name": "train_56_n32", "kind": "train", "n": 32, "size": 56, "classes": 100},
        # The benchmark's training step.
        {"name": "train_224_n32", "kind": "train", "n": 32, "size": 224, "classes": 1000},
        # One image at a time: a service that answers each request by itself.
        {"name": "infer_224_n1", "kind": "infer", "n": 1, "size": 224, "classes": 1000, "precision": "fp32"},
        # The benchmark's inference batch, in both precisions.
        {"name": "infer_224_n256", "kind": "infer", "n": 256, "size": 224, "classes": 1000, "precision": "fp32"},
        {"name": "infer_224_n256_bf16", "kind": "infer", "n": 256, "size": 224, "classes": 1000, "precision": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("conv", "pool", "small_net", "train", "infer"), (6, 1, 1, 2, 2))[0]
    if kind == "conv":
        while True:
            # channels of a network's inside are multiples of eight more often than not, its input has few
            c = rng.choice((_log_int(rng, 1, 512), 8 * _log_int(rng, 1, 64), 32 * _log_int(rng, 1, 16)))
            k = rng.choice((_log_int(rng, 1, 512), 8 * _log_int(rng, 1, 64), 32 * _log_int(rng, 1, 16)))
            r = rng.choice((1, 3, 3, 3, 5, 7))
            h = _log_int(rng, 7, 112)
            w = h if rng.random() < 0.6 else _log_int(rng, 7, 112)
            case = {"kind": "conv", "n": _log_int(rng, 1, 64), "c": c, "h": h, "w": w, "k": k, "r": r, "stride": rng.choice((1, 1, 2)),
                    "pad": rng.choice((r // 2, r // 2, 0)), "relu": rng.random() < 0.3,
                    "precision": "bf16" if rng.random() < 0.25 else "fp32"}
            if 2e7 <= work(case)["flops"] <= 3e10:
                return case
    if kind == "pool":
        k = rng.choice((2, 2, 3, 3, 5))
        while True:
            h = _log_int(rng, 7, 224)
            case = {"kind": "pool", "n": _log_int(rng, 1, 64), "c": _log_int(rng, 3, 512), "h": h,
                    "w": h if rng.random() < 0.5 else _log_int(rng, 7, 224), "k": k, "stride": rng.choice((k, 2, 1)),
                    "pad": rng.choice((0, k // 2))}
            if 1e5 <= work(case)["bytes"] <= 4e8:
                return case
    if kind == "small_net":
        return {"kind": "small_net", "n": _log_int(rng, 16, 1024), "size": rng.choice((28, rng.randint(20, 40))),
                "filters": rng.choice((8, 16, rng.randint(4, 32))), "graph": rng.random() < 0.5}
    size = rng.choice((56, 64, 96, 128, 160, 192, 224, rng.randint(56, 224), rng.randint(56, 224)))
    if kind == "train":
        n = _log_int(rng, 8, max(8, min(64, 32 * 224 * 224 // (size * size))))
        return {"kind": "train", "n": n, "size": size, "classes": rng.choice((10, 100, 1000))}
    n = _log_int(rng, 1, 256 if size < 200 else 128)
    return {"kind": "infer", "n": n, "size": size, "classes": rng.choice((10, 100, 1000)),
            "precision": rng.choice(("fp32", "bf16"))}


# --------------------------------------------------------------------------- device arrays and torch
class _Memory:
    """A device array's memory as torch takes it; torch keeps this object, and so the array, alive with its view."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str, "data": (array.ptr, False),
                                         "version": 2}


def _view(array):
    return torch.as_tensor(_Memory(array), device="cuda")


def _tensor(values, requires_grad=False):
    """A package tensor with a torch tensor's values (float32, or int64 labels), on the device."""
    array = be.empty(tuple(values.shape), np.int64 if values.dtype == torch.int64 else np.float32)
    be.synchronize()                             # whatever used this memory before has ended
    _view(array).copy_(values)
    torch.cuda.synchronize()
    return xs.Tensor(array, requires_grad=requires_grad)


def _outputs(state, arrays):
    """Torch views of ``arrays``.  Arrays that a program keeps from step to step (parameters, gradients) keep their
    memory: their views are made again only where the address has changed."""
    be.capi.flush_deferred()                     # reading a result makes the package launch what it held back
    kept = state.setdefault("views", {})
    out = []
    for i, a in enumerate(arrays):
        if i in kept and kept[i][0] == a.address() and kept[i][1].shape == a.shape:
            out.append(kept[i][1])
        else:
            v = _view(a)
            kept[i] = (a.address(), v)
            out.append(v)
    return out


# --------------------------------------------------------------------------- the networks
def _norm():
    """With shifts as a network in the middle of its training has them, not the zeros that it starts from."""
    return BatchNormalization(beta_initializer="normal")


class _Block(Module):
    def __init__(self, c_in, c_out, stride):
        super().__init__()
        self.body = Sequential(Conv2D(c_out, 3, stride=stride, padding=1, kernel_initializer="he_normal"), _norm(),
                               ReLU(True), Conv2D(c_out, 3, stride=1, padding=1, kernel_initializer="he_normal"),
                               _norm())
        self.shortcut = Sequential()
        if stride != 1 or c_in != c_out:
            self.shortcut = Sequential(Conv2D(c_out, 1, stride=stride, kernel_initializer="he_normal"), _norm())
        self.relu = ReLU(inplace=True)

    def forward(self, x, *args):
        out = self.body(x)
        out += self.shortcut(x)
        return self.relu(out)


class _ResNet18(Module):
    """Two blocks a stage, 7x7/2 stem, 3x3/2 max-pool, average over what is left of the image, one dense layer."""

    def __init__(self, classes, pool):
        super().__init__()
        self.stem = Sequential(Conv2D(64, 7, stride=2, padding=3, kernel_initializer="he_normal"), _norm(),
                               ReLU(inplace=True))
        self.pool = MaxPooling2D(kernel_size=3, stride=2, padding=1)
        blocks = []
        for c_in, c_out, stride in ((64, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 1), (128, 256, 2), (256, 256, 1),
                                    (256, 512, 2), (512, 512, 1)):
            blocks.append(_Block(c_in, c_out, stride))
        self.blocks = blocks
        self.stages = Sequential(*blocks)
        self.tail = Sequential(AvgPooling2D(pool), Flatten(), Dense(classes, kernel_initializer="he_normal"))

    def forward(self, x, *args):
        return self.tail(self.stages(self.pool(self.stem(x))))

    def sequences(self):
        blocks = [s for b in self.blocks for s in (b.body, b.shortcut, Sequential(b.relu))]
        return [self.stem, Sequential(self.pool)] + blocks + [self.tail]

    def trained(self):
        """The filters, the normalisations' scales and shifts and the dense layer, in the order of the forward.  Left out
        are the biases in front of a normalisation: it takes them away again and their gradient is rounding alone."""
        found = []
        for s in self.sequences():
            for layer in s._graph:
                p = [q for q in layer.parameters() if q is not None]
                found += p[:1] if isinstance(layer, Conv2D) else p
        return found


def _last_map(size):
    """Height of the last feature map of ResNet-18: five halvings, each rounded up."""
    for _ in range(5):
        size = (size + 1) // 2
    return size


# --------------------------------------------------------------------------- prepare, run
class _State(dict):
    """What a program keeps between passes.  Letting it go lets go of the layers' last outputs first: a layer, its output
    and its input refer to each other in a ring."""

    def __del__(self):
        net = self.get("net")
        parts = [net] if isinstance(net, Sequential) else [] if net is None else net.sequences()
        for s in parts:
            for layer in s._graph:
                if not isinstance(layer, Module):
                    layer.data = None


def prepare(case, seed):
    xs.GLOBAL.USE_CUDA = True
    xs.GLOBAL.TRAINING = True
    xs.GLOBAL.INPUTS = None
    np.random.seed(seed % (1 << 32))                     # the layers draw their parameters from it
    g = torch.Generator(device="cuda").manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=g, device="cuda")  # noqa: E731
    n = case["n"]
    state = _State(case=dict(case))
    if case["kind"] == "conv":
        c, k, r = case["c"], case["k"], case["r"]
        oh, ow = be.kernels.conv_out_hw(case["h"], case["w"], r, r, (case["stride"],) * 2, case["pad"])
        state["x"] = _tensor(normal(n, c, case["h"], case["w"]), True)
        state["w"] = xs.Parameter(_tensor(normal(k, c, r, r) * math.sqrt(2.0 / (c * r * r)), True))
        state["b"] = xs.Parameter(_tensor(normal(1, k) * 0.1, True))
        state["dy"] = _tensor(normal(n, k, oh, ow))
    elif case["kind"] == "pool":
        x = normal(n, case["c"], case["h"], case["w"])
        ties = torch.rand(x.shape, generator=g, device="cuda") < 0.05
        x = torch.where(ties, torch.roll(x, 1, 3), x)    # 5 % repeat their neighbour
        oh, ow = be.kernels.pool_out_hw(case["h"], case["w"], case["k"], (case["stride"],) * 2, case["pad"])
        state["x"] = _tensor(x, True)
        state["dy"] = _tensor(normal(n, case["c"], oh, ow))
    elif case["kind"] == "small_net":
        x = _tensor(normal(n, 1, case["size"], case["size"]))
        y = _tensor(torch.randint(0, 10, (n,), generator=g, device="cuda"))
        net = Sequential(Conv2D(case["filters"], 2, activation="relu", kernel_initializer="he_normal"), MaxPooling2D(2), Flatten(),
                         Dense(10))
        with xs.no_grad():
            net(x)                                       # creates the parameters
        xs.GLOBAL.INPUTS = None
        params = [p for layer in net._graph for p in layer.parameters() if p is not None]
        state.update(x=x, y=y, net=net, params=params, opt=SGD(params, lr=0.01), loss=xs.nn.CrossEntropyLoss())
        if case["graph"]:
            _step(state)                                 # the buffers a step needs exist before it is recorded
            state["step"] = xs.StepGraph()
            with state["step"].capture():
                state["recorded"] = _step(state)
            be.synchronize()
    else:
        x = _tensor(normal(n, 3, case["size"], case["size"]))
        net = _ResNet18(case["classes"], _last_map(case["size"])).to("cuda")
        with xs.no_grad():
            net(xs.Tensor(x.eval.leading(0, 1).copy()))  # creates the parameters
        xs.GLOBAL.INPUTS = None
        state.update(x=x, net=net)
        if case["kind"] == "train":
            state["y"] = _tensor(torch.randint(0, case["classes"], (n,), generator=g, device="cuda"))
            state.update(params=net.trained(), opt=SGD(list(net.parameters()), lr=0.01), loss=xs.nn.CrossEntropyLoss())
    return state


def _step(s):
    """One training step as a user's loop has it: the loss, the logits; gradients and parameters are updated in place."""
    s["opt"].zero_grad()
    logits = s["net"](s["x"])
    z = logits.eval
    loss = s["loss"](logits, s["y"])
    value = loss.eval
    loss.backward()
    s["opt"].step()
    return value, z


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "conv":
        x, w, b = state["x"], state["w"], state["b"]
        for t in (x, w, b):
            t.zero_grad()
        with xs.conv_precision(case["precision"]):
            y = F.conv2d(x, w, b, (case["stride"],) * 2, case["pad"], activation="relu" if case["relu"] else None)
            value = y.eval
            y.backward(state["dy"])
        return _outputs(state, [x.grad.eval, w.grad.eval, b.grad.eval, value])
    if kind == "pool":
        x = state["x"]
        x.zero_grad()
        y = F.max_pool2d(x, case["k"], (case["stride"],) * 2, case["pad"])
        value = y.eval
        y.backward(state["dy"])
        return _outputs(state, [x.grad.eval, value])
    if kind == "small_net" and case["graph"]:
        state["step"].replay()
        return _outputs(state, [p.eval for p in state["params"]] + list(state["recorded"]))
    if kind in ("small_net", "train"):
        xs.GLOBAL.TRAINING = True
        value, logits = _step(state)
        return _outputs(state, [p.eval for p in state["params"]] + [value, logits])
    xs.GLOBAL.TRAINING = False
    with xs.no_grad(), xs.conv_precision(case["precision"]):
        logits = state["net"](state["x"]).eval
    xs.GLOBAL.INPUTS = None
    return _outputs(state, [logits])


# --------------------------------------------------------------------------- what a pass cannot do without
def _resnet18_macs(size, classes):
    """(multiplications of all convolutions and the dense layer for one image, those of the first convolution, parameters)"""
    h = (size + 1) // 2
    stem = h * h * 64 * 3 * 49
    macs, params = stem, 64 * 3 * 49 + 3 * 64
    h = (h + 1) // 2
    for c_in, c_out, stride in ((64, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 1), (128, 256, 2), (256, 256, 1), (256, 512, 2),
                                (512, 512, 1)):
        h = (h + stride - 1) // stride
        macs += h * h * c_out * 9 * (c_in + c_out)
        params += c_out * 9 * (c_in + c_out) + 6 * c_out
        if stride != 1:
            macs += h * h * c_out * c_in
            params += c_out * c_in + 3 * c_out
    return macs + 512 * classes, stem, params + 513 * classes


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "conv":
        oh = (case["h"] + 2 * case["pad"] - case["r"]) // case["stride"] + 1
        ow = (case["w"] + 2 * case["pad"] - case["r"]) // case["stride"] + 1
        if oh < 1 or ow < 1:
            return {"bytes": 0, "flops": 0}
        taps = case["c"] * case["r"] ** 2
        x, y, w = n * case["c"] * case["h"] * case["w"], n * case["k"] * oh * ow, case["k"] * (taps + 1)
        return {"bytes": 4 * 2 * (x + y + w), "flops": 3 * 2 * n * oh * ow * case["k"] * taps}
    if kind == "pool":
        oh = (case["h"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1
        ow = (case["w"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1
        if oh < 1 or ow < 1:
            return {"bytes": 0, "flops": 0}
        return {"bytes": 4 * 2 * n * case["c"] * (case["h"] * case["w"] + oh * ow), "flops": n * case["c"] * oh * ow * case["k"] ** 2}
    if kind == "small_net":
        s, f = case["size"], case["filters"]
        conv, flat = (s - 1) * (s - 1) * f * 4, ((s - 1) // 2) ** 2 * f
        params = 5 * f + 10 * flat + 10
        return {"bytes": 4 * (n * s * s + 2 * params + 10 * n) + 8 * n, "flops": 2 * n * (2 * conv + 3 * 10 * flat)}
    macs, stem, params = _resnet18_macs(case["size"], case["classes"])
    images = 4 * n * 3 * case["size"] ** 2
    if kind == "train":
        return {"bytes": images + 4 * (2 * params + n * case["classes"]), "flops": 2 * n * (3 * macs - stem)}
    return {"bytes": images + 4 * (params + n * case["classes"]), "flops": 2 * n * macs}


def tolerance(case):
    """Each figure is about four times what the same path gave on the same inputs with its sums in another order."""
    if case["kind"] == "pool":
        return "exact"                                   # a choice of values, and sums in a fixed order
    if case["kind"] in ("small_net", "train"):
        # three steps: a sum within rounding of zero falls on the other side of a ReLU, or another value wins its window
        return {"rel": 4e-4, "max": 4e-3}
    if case["precision"] == "bf16":
        return {"rel": 5e-3, "max": 3e-2}                # a value stored as bf16 may round the other way
    return {"rel": 3e-6, "max": 3e-5}


# --------------------------------------------------------------------------- the same in 64 bits, by torch alone
def _double(array):
    return _view(array).double()


def _exact_layer(layer, x, p, training):
    if isinstance(layer, Module):
        return _exact_net(layer, x, p, training)
    if isinstance(layer, Conv2D):
        w = p(layer._parameters[0])
        x = torch.nn.functional.conv2d(x, w, p(layer._parameters[1]).reshape(-1), layer.stride, layer.pad_size)
        return x.relu() if layer.activation is not None else x
    if isinstance(layer, BatchNormalization):
        gamma, beta = (p(q).reshape(1, -1, 1, 1) for q in layer._parameters)
        if training:
            mean, var = x.mean((0, 2, 3), keepdim=True), x.var((0, 2, 3), unbiased=False, keepdim=True)
        else:
            mean, var = (_double(q.eval).reshape(1, -1, 1, 1) for q in (layer.moving_mean, layer.moving_variance))
        return (x - mean) / torch.sqrt(var + layer.epsilon) * gamma + beta
    if isinstance(layer, ReLU):
        return x.relu()
    if isinstance(layer, MaxPooling2D):
        k, pad = layer.kernel_size, layer.padding
        k = k if isinstance(k, int) else k[0]
        x = torch.nn.functional.pad(x, (pad,) * 4)           # border cells compete with their zeros
        return torch.nn.functional.max_pool2d(x, k, layer.stride)
    if isinstance(layer, AvgPooling2D):
        return x.mean((2, 3), keepdim=True)                  # the window is the whole map
    if isinstance(layer, Flatten):
        return x.flatten(1)
    return x @ p(layer._parameters[0]) + p(layer._parameters[1])


def _exact_seq(seq, x, p, training):
    for layer in seq._graph or []:
        x = _exact_layer(layer, x, p, training)
    return x


def _exact_net(net, x, p, training):
    if isinstance(net, _Block):
        return (_exact_seq(net.body, x, p, training) + _exact_seq(net.shortcut, x, p, training)).relu()
    if isinstance(net, _ResNet18):
        x = _exact_layer(net.pool, _exact_seq(net.stem, x, p, training), p, training)
        return _exact_seq(net.tail, _exact_seq(net.stages, x, p, training), p, training)
    return _exact_seq(net, x, p, training)


def exact(case, seed):
    """What ``run`` returns for these inputs, computed by torch in 64 bits."""
    state = prepare(case, seed)
    kind = case["kind"]
    with torch.backends.cudnn.flags(enabled=False):          # torch's own convolution takes 64 bits
        if kind == "conv":
            x, w, b = (_double(state[q].eval).requires_grad_() for q in ("x", "w", "b"))
            y = torch.nn.functional.conv2d(x, w, b.reshape(-1), (case["stride"],) * 2, case["pad"])
            y = y.relu() if case["relu"] else y
            grads = torch.autograd.grad(y, (x, w, b), _double(state["dy"].eval))
            return [*grads, y.detach()]
        if kind == "pool":
            x = _double(state["x"].eval).requires_grad_()
            y = torch.nn.functional.max_pool2d(torch.nn.functional.pad(x, (case["pad"],) * 4), case["k"], case["stride"])
            return [torch.autograd.grad(y, x, _double(state["dy"].eval))[0], y.detach()]
        held = {}

        def p(parameter):
            if id(parameter) not in held:
                held[id(parameter)] = _double(parameter.eval).requires_grad_(kind != "infer")
            return held[id(parameter)]

        x = _double(state["x"].eval)
        if kind == "infer":
            with torch.no_grad():
                parts = 4 if case["n"] >= 64 else 1          # the unfolded images of a whole batch are many
                return [torch.cat([_exact_net(state["net"], part, p, False) for part in x.chunk(parts)])]
        logits = _exact_net(state["net"], x, p, True)
        loss = torch.nn.functional.cross_entropy(logits, _view(state["y"].eval).reshape(-1))
        params = [p(q) for q in state["params"]]
        grads = torch.autograd.grad(loss, params)
        return [(q - 0.01 * g).detach() for q, g in zip(params, grads)] + [loss.detach().reshape(1), logits.detach()]
