"""What a user of this package has it do, as cases that can be timed: `listed()` names them, `draw()` makes more of the
same kinds and ranges, `prepare()` makes what a program has in hand before the call and `run()` is one pass.

The kinds:
  linear   a fully connected layer through execute_graph: relu(x w + b) and its column sums, or forward and backward
  mlp      one SGD step of a two-layer perceptron in f32 (a small training loop, bound by latency)
  cell     the fused product with its 40-op epilogue (configs.c4_graph), one kernel on the caller's buffers
  planned  a product with operand and result arithmetic, split into kernels by the fusion search
  permute  PermuteDims on the caller's buffers
  chain    a pointwise chain and reductions of its values (configs.c3_chain), one kernel on the caller's buffers
  infer    an image classifier from a batch in host memory to probabilities in host memory
  train    one SGD step of that classifier; its results are the next step's inputs
"""
import ctypes
import functools
import math

import numpy as np
import torch

import helium_amd as ha
from helium_amd import configs, fusion_search
from helium_amd.backend import Tensor, execute_graph

LEARNING_RATE = 0.01
BN_EPSILON = 1e-3
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "bf16": 2}


def listed():
    return [
        # the smallest graph worth a call: a 256 x 512 activation through one f32 layer (configs.c1_ir_graph's size)
        {"name": "linear_f32", "kind": "linear", "rows": 256, "inner": 512, "cols": 512, "dtype": "f32", "backward": False},
        # a layer's forward and backward pass in mixed precision at sizes no tile divides
        {"name": "linear_bf16_ragged", "kind": "linear", "rows": 1537, "inner": 1000, "cols": 777, "dtype": "bf16", "backward": True},
        # a training step on digit-sized images: some twenty small operations, each far from filling the chip
        {"name": "mlp_step", "kind": "mlp", "batch": 64, "inner": 784, "hidden": 512, "classes": 10},
        # the benchmark's headline product, storing the gradients that the next products read
        {"name": "cell_4096", "kind": "cell", "size": 4096, "full": True},
        # a batch of middling products whose rows start at odd addresses
        {"name": "planned_ragged", "kind": "planned", "batch": 4, "m": 777, "k": 1000, "n": 1203},
        # an activation changes layout
        {"name": "permute_nhwc_bf16", "kind": "permute", "shape": "64,56,56,256", "perm": "0,3,1,2", "dtype": "bf16"},
        # the same in f32 at odd extents
        {"name": "permute_ragged_f32", "kind": "permute", "shape": "37,101,53,67", "perm": "0,3,1,2", "dtype": "f32"},
        # a swap of outermost and innermost dim that no cache holds
        {"name": "permute_large_f32", "kind": "permute", "shape": "1024,128,128,32", "perm": "3,1,2,0", "dtype": "f32"},
        # pointwise arithmetic over rows of odd length: its values and two reductions of them
        {"name": "chain_ragged", "kind": "chain", "rows": 5000, "cols": 3001, "bias_axis": 2, "full": True},
        # serving one image: the latency of a whole network, host memory to host memory
        {"name": "infer_one", "kind": "infer", "batch": 1, "image": 224, "width": 32, "classes": 1000},
        # a training step at the size the parity tests take, bound by launches
        {"name": "train_small", "kind": "train", "batch": 8, "image": 64, "width": 32, "classes": 1000},
        # a training step at the benchmark's batch and image size
        {"name": "train_large", "kind": "train", "batch": 128, "image": 224, "width": 32, "classes": 1000},
    ]


def _log(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["linear"] * 3 + ["mlp"] * 2 + ["cell"] + ["planned"] * 2 + ["permute"] * 3 + ["chain"] * 2 + ["infer", "train"])
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 16, 8192), "inner": _log(rng, 32, 4096), "cols": _log(rng, 10, 4096),
                "dtype": rng.choice(["f32", "bf16", "bf16"]), "backward": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 16, 1024), "inner": _log(rng, 32, 2048), "hidden": _log(rng, 32, 2048), "classes": _log(rng, 2, 1000)}
    if kind == "cell":
        size = _log(rng, 256, 4096)
        return {"kind": kind, "size": size if rng.random() < 0.5 else size // 64 * 64, "full": rng.random() < 0.5}
    if kind == "planned":
        return {"kind": kind, "batch": _log(rng, 1, 16), "m": _log(rng, 64, 2048), "k": _log(rng, 64, 2048), "n": _log(rng, 64, 2048)}
    if kind == "permute":
        numel, rank = _log(rng, 1 << 20, 1 << 28), rng.randint(2, 5)
        parts = [rng.uniform(0.4, 1.6) for _ in range(rank)]
        shape = [max(2, round(numel ** (p / sum(parts)))) for p in parts]
        if rng.random() < 0.5:
            shape = [max(8, -(-d // 8) * 8) if d > 8 else d for d in shape]
        perm = list(range(rank))
        while perm == sorted(perm):
            rng.shuffle(perm)
        return {"kind": kind, "shape": ",".join(map(str, shape)), "perm": ",".join(map(str, perm)), "dtype": rng.choice(["f32", "bf16"])}
    if kind == "chain":
        return {"kind": kind, "rows": _log(rng, 16, 8192), "cols": _log(rng, 16, 8192), "bias_axis": rng.choice([1, 2]), "full": rng.random() < 0.5}
    case = {"kind": kind, "width": rng.choice([16, 24, 32]), "classes": _log(rng, 10, 1000)}
    if kind == "infer":
        return {**case, "batch": _log(rng, 1, 64), "image": _log(rng, 32, 224)}
    return {**case, "batch": _log(rng, 4, 128), "image": _log(rng, 32, 224)}


# ---- tensors ---------------------------------------------------------------------------------------------------
class _View:
    """Storage of this package as torch sees it; torch keeps the object, and so the storage, while it has a view."""

    def __init__(self, tensor, shape, dtype):
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": {"f32": "<f4", "bf16": "<i2"}[dtype],
                                         "data": (tensor.ptr.value, False), "version": 3}


class Outputs(dict):
    """A graph's results by name, each {tensor, shape, dtype}; reading an entry gives a torch view of the tensor."""

    def __getitem__(self, name):
        tensor, shape, dtype = dict.__getitem__(self, name)
        return torch.as_tensor(_View(tensor, shape, dtype), device="cuda").view(TORCH[dtype])


class _Pointer:
    """A torch tensor's memory as the package takes buffers."""

    def __init__(self, tensor):
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _host(x, dtype):
    """A torch tensor in the package's storage form, in host memory."""
    x = x.to(TORCH[dtype]).cpu().contiguous()
    return (x.view(torch.int16) if dtype == "bf16" else x).numpy().view(np.uint16 if dtype == "bf16" else np.float32)


def _device(x, dtype):
    return Tensor.from_numpy(_host(x, dtype), dtype, x.numel())


def _normal(gen, shape, scale=1.0):
    return torch.randn(list(shape), generator=gen, device="cuda") * scale


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


# ---- graphs ----------------------------------------------------------------------------------------------------
class _Graph:
    """A recorded graph with names for its inputs and outputs: name -> (node, shape, dtype)."""

    def __init__(self):
        self.g, self.inputs, self.outputs, self.updates = ha.ir.OpGraph(), {}, {}, {}

    def input(self, name, shape, dtype="f32"):
        node = self.g.new_input(list(shape), dtype)
        self.inputs[name] = (node, tuple(shape), dtype)
        return node

    def output(self, name, node):
        shape, dtype = self.g.descriptor(node)
        self.outputs[name] = (self.g.new_output(node), tuple(shape), dtype)

    def shape(self, node):
        return self.g.descriptor(node)[0]

    def const(self, value, like):
        return self.g.constant(value, "f32", self.shape(like))

    def mul(self, a, b):
        return self.g.binary(a, b, "mul")

    def add(self, a, b):
        return self.g.binary(a, b, "add")

    def sub(self, a, b):
        return self.g.binary(a, self.g.unary(b, "neg"), "add")

    def scale(self, x, value):
        return self.mul(x, self.const(value, x))

    def update(self, name, gradient):
        """Plain gradient descent: the new value of an input is an output of the same name."""
        w = self.inputs[name][0]
        self.output(name, self.sub(w, self.scale(gradient, LEARNING_RATE)))
        self.updates[self.inputs[name][0]] = name

    def feed(self, name, node):
        """An output that replaces an input on the next pass."""
        self.output(name, node)
        self.updates[self.inputs[name][0]] = name

    def rows(self, v, like):
        """[cols] -> [rows, cols]"""
        return self.g.broadcast(v, 2, [(0, self.shape(like)[0])])

    def columns(self, v, like):
        """[rows, 1] -> [rows, cols]"""
        return self.g.broadcast(v, 2, [(1, self.shape(like)[1])])

    def row_sum(self, x):
        """Sum over the rows: [rows, cols] -> [cols]"""
        return self.g.reshape(self.g.reduce(self.g.swap_dims(x, 0, 1), "sum", 1), [self.shape(x)[1]])

    def softmax_cross_entropy(self, logits, labels):
        """Returns (loss [1, 1], probabilities, gradient of the mean loss)."""
        g, n = self.g, self.shape(logits)[0]
        shifted = self.sub(logits, self.columns(g.reduce(logits, "max", 1), logits))
        total = g.reduce(g.unary(shifted, "exp"), "sum", 1)
        log_p = self.sub(shifted, self.columns(g.unary(total, "log"), logits))
        probs = g.unary(log_p, "exp")
        loss = self.scale(g.reduce(self.mul(labels, log_p), "sum", 2), -1.0 / n)
        return loss, probs, self.scale(self.sub(probs, labels), 1.0 / n)

    def masked(self, flow, x):
        """The flow where x is above zero."""
        zero = self.const(0.0, flow)
        return self.g.select(zero, flow, self.g.compare(x, self.const(0.0, x), "gt"))


@functools.lru_cache(maxsize=None)
def _linear_graph(rows, inner, cols, dtype, backward):
    G = _Graph()
    g, precision = G.g, "f32_f32" if dtype == "f32" else "bf16_f32"
    x, w, b = G.input("x", [rows, inner], dtype), G.input("w", [inner, cols], dtype), G.input("b", [cols])
    y = g.unary(G.add(g.matmul(x, w, precision), G.rows(b, x)), "relu")
    G.output("y", g.change_data_type(y, dtype))
    if not backward:
        G.output("sums", G.row_sum(y))
        return G
    flow = G.input("flow", [rows, cols], dtype)
    f = G.masked(g.change_data_type(flow, "f32"), y)
    f16 = g.change_data_type(f, dtype)
    G.output("dx", g.change_data_type(g.matmul(f16, g.swap_dims(w, 0, 1), precision), dtype))
    G.output("dw", g.matmul(g.swap_dims(x, 0, 1), f16, precision))
    G.output("db", G.row_sum(f))
    return G


@functools.lru_cache(maxsize=None)
def _mlp_graph(batch, inner, hidden, classes):
    G = _Graph()
    g = G.g
    x, labels = G.input("x", [batch, inner]), G.input("labels", [batch, classes])
    w1, b1 = G.input("w1", [inner, hidden]), G.input("b1", [hidden])
    w2, b2 = G.input("w2", [hidden, classes]), G.input("b2", [classes])
    h = g.unary(G.add(g.matmul(x, w1, "f32_f32"), G.rows(b1, x)), "relu")
    logits = G.add(g.matmul(h, w2, "f32_f32"), G.rows(b2, x))
    loss, _, d = G.softmax_cross_entropy(logits, labels)
    dh = G.masked(g.matmul(d, g.swap_dims(w2, 0, 1), "f32_f32"), h)
    G.output("loss", loss)
    G.update("w2", g.matmul(g.swap_dims(h, 0, 1), d, "f32_f32"))
    G.update("b2", G.row_sum(d))
    G.update("w1", g.matmul(g.swap_dims(x, 0, 1), dh, "f32_f32"))
    G.update("b1", G.row_sum(dh))
    return G


class _Classifier(_Graph):
    """A residual image classifier on NHWC bf16 activations with f32 parameters: a 7x7 stride-2 convolution, four blocks
    that halve the extents and double the channels, batch norm, global average pooling and a linear layer."""

    def __init__(self, batch, image, width, classes, train):
        super().__init__()
        self.train = train
        x = self.input("image", [batch, image, image, 3], "bf16")
        backs = []
        x, back = self.conv("head", x, width, 7, 2, flow_needed=False)
        backs.append(back)
        for k in range(4):
            x, back = self.block("block%d" % k, x, width << (k + 1))
            backs.append(back)
        x, back = self.bn_relu("tail_bn", x)
        backs.append(back)
        logits, back = self.pooled_linear(x, classes)
        backs.append(back)
        if not train:
            total = lambda v, fn: self.columns(self.g.reduce(v, fn, 1), logits)  # noqa: E731
            e = self.g.unary(self.sub(logits, total(logits, "max")), "exp")
            self.output("probs", self.mul(e, self.g.unary(total(e, "sum"), "recip")))
            return
        loss, probs, flow = self.softmax_cross_entropy(logits, self.input("labels", [batch, classes]))
        self.output("loss", loss)
        self.output("probs", probs)
        for back in reversed(backs):
            flow = back(flow)

    def cast(self, x, dtype):
        return self.g.change_data_type(x, dtype)

    def channels(self, v, like):
        """[c] -> the shape of an activation"""
        return self.g.broadcast(v, 4, list(enumerate(self.shape(like)[:3])))

    def over_pixels(self, x, fn):
        """An activation reduced over everything but its channels."""
        return self.g.reshape(self.g.reduce(self.g.swap_dims(x, 0, 3), fn, 3), [self.shape(x)[3]])

    def conv(self, name, x, out_channels, kernel, stride=1, flow_needed=True):
        _, h, w, c = self.shape(x)
        params = {"in_channels": c, "out_channels": out_channels, "kernel_size": [kernel, kernel], "stride": [stride, stride]}
        weights = self.cast(self.input(name, [out_channels, kernel, kernel, c]), "bf16")

        def back(flow):
            self.update(name, self.cast(self.g.conv_backward_filter(flow, x, params), "f32"))
            return self.g.conv_backward_data(flow, weights, params, [h, w]) if flow_needed else None

        return self.g.conv(x, weights, params), back

    def bn_relu(self, name, x):
        g, c = self.g, self.shape(x)[3]
        mean, var, scale, bias = (self.input(name + "." + p, [c]) for p in ("mean", "var", "scale", "bias"))
        x = self.cast(x, "f32")
        if self.train:
            running = mean, var
            mean = self.over_pixels(x, "mean")
            var = self.sub(self.over_pixels(self.mul(x, x), "mean"), self.mul(mean, mean))
            for part, old, new in zip(("mean", "var"), running, (mean, var)):
                self.feed(name + "." + part, self.add(self.scale(old, 0.9), self.scale(new, 0.1)))
        inverse = g.unary(g.unary(self.add(var, self.const(BN_EPSILON, var)), "sqrt"), "recip")
        normal = self.mul(self.sub(x, self.channels(mean, x)), self.channels(inverse, x))
        y = self.add(self.mul(normal, self.channels(scale, x)), self.channels(bias, x))

        def back(flow):
            f = self.masked(self.cast(flow, "f32"), y)
            sum_f, sum_fn = self.over_pixels(f, "sum"), self.over_pixels(self.mul(f, normal), "sum")
            self.update(name + ".scale", sum_fn)
            self.update(name + ".bias", sum_f)
            b, h, w, _ = self.shape(x)
            share = lambda v: self.channels(self.scale(v, 1.0 / (b * h * w)), x)  # noqa: E731
            centred = self.sub(self.sub(f, share(sum_f)), self.mul(normal, share(sum_fn)))
            return self.cast(self.mul(centred, self.channels(self.mul(scale, inverse), x)), "bf16")

        return self.cast(g.unary(y, "relu"), "bf16"), back

    def block(self, name, x, out_channels):
        x, bn1 = self.bn_relu(name + ".bn1", x)
        shortcut, side = self.conv(name + ".shortcut", x, out_channels, 1, 2)
        h, conv1 = self.conv(name + ".conv1", x, out_channels, 3, 2)
        h, bn2 = self.bn_relu(name + ".bn2", h)
        h, conv2 = self.conv(name + ".conv2", h, out_channels, 3)
        return self.add(h, shortcut), lambda flow: bn1(self.add(conv1(bn2(conv2(flow))), side(flow)))

    def pooled_linear(self, x, classes):
        g = self.g
        b, h, w, c = self.shape(x)
        pooled = g.reshape(g.reduce(g.swap_dims(g.swap_dims(self.cast(x, "f32"), 2, 3), 1, 2), "mean", 2), [b, c])
        pooled = self.cast(pooled, "bf16")
        weights = self.cast(self.input("linear", [c, classes]), "bf16")
        bias = self.input("linear.bias", [classes])

        def back(flow):
            self.update("linear.bias", self.row_sum(flow))
            flow = self.cast(flow, "bf16")
            self.update("linear", g.matmul(g.swap_dims(pooled, 0, 1), flow, "bf16_f32"))
            d = self.scale(g.matmul(flow, g.swap_dims(weights, 0, 1), "bf16_f32"), 1.0 / (h * w))
            return g.broadcast(g.reshape(self.cast(d, "bf16"), [b, 1, 1, c]), 4, [(1, h), (2, w)])

        return self.add(g.matmul(pooled, weights, "bf16_f32"), self.rows(bias, pooled)), back


@functools.lru_cache(maxsize=None)
def _classifier(batch, image, width, classes, train):
    return _Classifier(batch, image, width, classes, train)


def _values(gen, name, shape):
    """Parameters as a training run holds them: scaled weights, statistics and factors near their starting values."""
    if name == "labels":
        return torch.nn.functional.one_hot(torch.randint(0, shape[1], (shape[0],), generator=gen, device="cuda"), shape[1]).float()
    if name.endswith(".var") or name.endswith(".scale"):
        return torch.rand(shape, generator=gen, device="cuda") * 0.5 + 0.75
    if name.endswith(".mean") or name.endswith("bias") or name in ("b", "b1", "b2"):
        return _normal(gen, shape, 0.1)
    if len(shape) == 4 and name != "image":
        return _normal(gen, shape, (2.0 / (shape[1] * shape[2] * shape[3])) ** 0.5)
    if name in ("w", "w1", "w2", "linear"):
        return _normal(gen, shape, shape[0] ** -0.5)
    return _normal(gen, shape)


@functools.lru_cache(maxsize=None)
def _planned(batch, m, k, n):
    g = ha.fusion.OpGraph()
    a, t, b = g.producer([batch, m, k]), g.producer([batch, m, k]), g.producer([batch, k, n])
    bias = g.producer([batch, 1, n], "f32")
    product = g.matmul(g.binary(g.unary(a, "relu"), t, "mul"), b)
    y = g.consumer(g.unary(g.binary(product, g.broadcast(bias, 1, m), "add"), "relu"))
    plan = fusion_search.FusionPlan(g, fusion_search.MIN_MI355X_COST)
    plan.precompile()
    return plan, [(a, [batch, m, k], "bf16"), (t, [batch, m, k], "bf16"), (b, [batch, k, n], "bf16"), (bias, [batch, 1, n], "f32")], y


@functools.lru_cache(maxsize=None)
def _kernel(kind, *args):
    """A kernel that runs on the caller's buffers, and its graph."""
    if kind == "cell":
        g, _ = configs.c4_graph(args[0], full_size_outputs=args[1])
        return ha.TileKernel.fused(g), g
    g, _, outs = configs.c3_chain(args[0], args[1], bias_axis=args[2], make_inputs=False)
    if args[3]:
        g.consumer(outs["r"], "f32")
    return ha.TileKernel.auxiliary(g), g


@functools.lru_cache(maxsize=None)
def _permute(shape, perm, dtype):
    return ha.PermuteDims([int(d) for d in shape.split(",")], dtype, perm=[int(p) for p in perm.split(",")])


def _graph_of(case):
    if case["kind"] == "linear":
        return _linear_graph(case["rows"], case["inner"], case["cols"], case["dtype"], case["backward"])
    if case["kind"] == "mlp":
        return _mlp_graph(case["batch"], case["inner"], case["hidden"], case["classes"])
    return _classifier(case["batch"], case["image"], case["width"], case["classes"], case["kind"] == "train")


# ---- passes ----------------------------------------------------------------------------------------------------
def prepare(case, seed):
    ha.device.init()
    gen, kind = _generator(seed), case["kind"]
    if kind == "permute":
        op = _permute(case["shape"], case["perm"], case["dtype"])
        src = _normal(gen, op.shape).to(TORCH[case["dtype"]])
        out = torch.empty(op.out_shape, dtype=src.dtype, device="cuda")
        return {"kind": kind, "op": op, "src": src, "out": out, "addresses": (src.data_ptr(), out.data_ptr())}
    if kind in ("cell", "chain"):
        kernel, g = _kernel(kind, case["size"], case["full"]) if kind == "cell" else _kernel(kind, case["rows"], case["cols"], case["bias_axis"], case["full"])
        shapes = {n["id"]: n["shape"] for n in g.nodes}
        buffers, outs = [], {}
        for a in kernel.args:
            shape, dtype = shapes[a["node"]], TORCH[a["dtype"]]
            if a["is_output"]:
                outs[str(a["node"])] = torch.empty(shape, dtype=dtype, device="cuda")
                buffers.append(outs[str(a["node"])])
                continue
            if kind == "chain":
                x = torch.rand(shape, generator=gen, device="cuda") * 2 - 1
            else:  # operands of the product, other products' results, state and biases (configs.c4_inputs)
                x = _normal(gen, shape, 0.02 if a["node"] in (1, 2) else 0.02 * 0.02 * case["size"] ** 0.5 if a["node"] in (13, 24, 26) else 1.0)
            buffers.append(x.to(dtype))
        return {"kind": kind, "kernel": kernel, "buffers": buffers, "addresses": [b.data_ptr() for b in buffers], "outs": outs}
    if kind == "planned":
        plan, inputs, y = _planned(case["batch"], case["m"], case["k"], case["n"])
        scale = dict(zip([i[0] for i in inputs], (1.0, 1.0, case["k"] ** -0.5, 1.0)))
        tensors = {n: _normal(gen, shape, scale[n]).to(TORCH[dtype]) for n, shape, dtype in inputs}
        out = torch.empty([case["batch"], case["m"], case["n"]], dtype=torch.bfloat16, device="cuda")
        return {"kind": kind, "plan": plan, "tensors": tensors, "out": out, "producers": {n: _Pointer(t) for n, t in tensors.items()},
                "consumers": {y: _Pointer(out)}}
    G = _graph_of(case)
    state = {"kind": kind, "G": G, "tensors": {}}
    for name, (node, shape, dtype) in G.inputs.items():
        x = _values(gen, name, shape)
        if kind == "infer" and name == "image":
            state["image"], state["image_node"] = _host(x, dtype), node
        else:
            state["tensors"][node] = _device(x, dtype)
    return state


def run(state):
    kind = state["kind"]
    if kind == "permute":
        state["op"].execute(*state["addresses"])
        return state["out"]
    if kind in ("cell", "chain"):
        state["kernel"].execute(state["addresses"])
        return state["outs"]
    if kind == "planned":
        state["plan"].execute(state["producers"], state["consumers"])
        return state["out"]
    G, tensors = state["G"], state["tensors"]
    if kind == "infer":
        tensors = {**tensors, state["image_node"]: Tensor.from_numpy(state["image"], "bf16")}
    results = execute_graph(G.g, tensors)
    if kind == "infer":
        node, shape, _ = G.outputs["probs"]
        return results[node].to_numpy().reshape(shape)
    for node, name in G.updates.items():
        tensors[node] = results[G.outputs[name][0]]
    return Outputs({name: (results[node], shape, dtype) for name, (node, shape, dtype) in G.outputs.items()})


# ---- what a pass cannot do without -----------------------------------------------------------------------------
def _conv_flops(case):
    """Multiply-adds of the classifier's convolutions and its linear layer, times two; backward costs twice forward
    (the head's image needs no gradient)."""
    b, w, extent, train = case["batch"], case["width"], -(-case["image"] // 2), case["kind"] == "train"
    total = 2.0 * b * extent * extent * w * 49 * 3 * (2 if train else 1)
    for k in range(4):
        c, extent = w << k, -(-extent // 2)
        total += 2.0 * b * extent * extent * 2 * c * (c + 9 * c + 9 * 2 * c) * (3 if train else 1)
    return total + 2.0 * b * (w << 4) * case["classes"] * (3 if train else 1)


def work(case):
    kind = case["kind"]
    if kind == "permute":
        return {"bytes": 2 * SIZE[case["dtype"]] * math.prod(int(d) for d in case["shape"].split(",")), "flops": 0}
    if kind == "chain":
        r, c = case["rows"], case["cols"]
        return {"bytes": 4 * ((5 if case["full"] else 4) * r * c + (r if case["bias_axis"] == 2 else c) + 1 + c), "flops": 0}
    if kind == "cell":
        n = case["size"]
        return {"bytes": (7 + (2 if case["full"] else 0)) * 2 * n * n + 4 * (4 * n + 1), "flops": 2.0 * n ** 3}
    if kind == "planned":
        b, m, k, n = (case[v] for v in ("batch", "m", "k", "n"))
        return {"bytes": b * (2 * (2 * m * k + k * n + m * n) + 4 * n), "flops": 2.0 * b * m * n * k}
    G = _graph_of(case)
    moved = sum(math.prod(shape) * SIZE[dtype] for table in (G.inputs, G.outputs) for _, shape, dtype in table.values())
    if kind == "linear":
        return {"bytes": moved, "flops": 2.0 * case["rows"] * case["inner"] * case["cols"] * (3 if case["backward"] else 1)}
    if kind == "mlp":
        b, i, h, c = (case[v] for v in ("batch", "inner", "hidden", "classes"))
        return {"bytes": moved, "flops": 2.0 * b * h * (2 * i + 3 * c)}
    return {"bytes": moved, "flops": _conv_flops(case)}


def tolerance(case):
    """Permutes move bits. 32-bit sums agree to 1e-5. Where values of 16 bits are rounded, another order of the sums moves
    some of them to the neighbouring value (2^-8), and a network carries that on from layer to layer."""
    kind = case["kind"]
    if kind == "permute":
        return "exact"
    if kind in ("chain", "mlp") or (kind == "linear" and case["dtype"] == "f32"):
        return {"rel": 1e-5, "max": 1e-2}
    return {"rel": 1e-2 if kind != "train" else 2e-2, "max": 0.5}
