"""The work that a program built on ferrograd_amd has the MI355X do, as
measurable cases: the tensor calls of the benchmark, the layers of the MLPs it
trains, and whole forward passes and train steps, from one image to the widest
batch. Every case goes through the public Python API (Tensor, Linear, Sgd and
the train loops of ferrograd_amd.mlp).

Inputs are drawn on the GPU from the seed alone, brought to the host as a
program's data is, and uploaded by Tensor.new / Tensor.write in prepare().
Outputs are views of the framework's own device buffers."""
from __future__ import annotations

import math

import torch

import ferrograd_amd as fg
from ferrograd_amd import Linear, Sgd, Tensor
from ferrograd_amd.mlp import Mlp, train_batches_native, train_step

LR = 0.01


def listed():
    return [
        # One image through the 784-128-10 classifier: the smallest call, launches and host latency.
        {"name": "classify_1", "kind": "forward", "batch": 1, "dims": "784,128,10"},
        # The 10,000-image test set through the same classifier, as each epoch's accuracy is measured.
        {"name": "classify_10000", "kind": "forward", "batch": 10000, "dims": "784,128,10"},
        # Fused elementwise arithmetic on vectors far larger than any cache.
        {"name": "pointwise_2p26", "kind": "pointwise", "n": 1 << 26},
        # Row sums of a fused elementwise expression.
        {"name": "row_sum_4096x4096", "kind": "row_sum", "rows": 4096, "cols": 4096},
        # Sums over the samples of a data set of 60,000 images (per-pixel means; a bias gradient).
        {"name": "col_sum_60000x784", "kind": "col_sum", "rows": 60000, "cols": 784},
        # One number from a whole tensor: the squared error of a prediction.
        {"name": "squared_error_5000x3001", "kind": "squared_error", "rows": 5000, "cols": 3001},
        # A transposed copy with odd sides.
        {"name": "transpose_4000x3001", "kind": "transpose", "rows": 4000, "cols": 3001, "dtype": "f32"},
        # Cross-entropy over a thousand classes and its gradient: the head of a larger classifier.
        {"name": "cross_entropy_4096x1000", "kind": "cross_entropy", "batch": 4096, "classes": 1000},
        # Linear forward, 4096 on every side.
        {"name": "linear_4096", "kind": "linear", "batch": 4096, "inputs": 4096, "outputs": 4096},
        # Linear forward and backward (input, weight and bias gradients) with ragged sides.
        {"name": "linear_grad_3000x1500x1001", "kind": "linear_grad", "batch": 3000, "inputs": 1500, "outputs": 1001},
        # Fifty train steps of the 784-128-10 classifier over a resident data set, batches of 256.
        {"name": "train_loop_256", "kind": "train_loop", "batch": 256, "dims": "784,128,10", "steps": 50},
        # One train step of the wide MLP at batch 8192.
        {"name": "train_step_8192", "kind": "train_step", "batch": 8192, "dims": "784,4096,4096,10"},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm; any remainder comes up."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "pointwise", "row_sum", "col_sum", "squared_error", "transpose", "cross_entropy",
                       "linear", "linear", "linear_grad", "train_loop", "train_step"])
    case = {"kind": kind}
    if kind == "forward":
        case["batch"] = _log_int(rng, 1, 20000)
        case["dims"] = "784,%d,%d" % (_log_int(rng, 32, 2048), rng.choice([2, 10, 10, 37, 100]))
    elif kind == "pointwise":
        case["n"] = _log_int(rng, 64, 1 << 26)
    elif kind in ("row_sum", "col_sum", "squared_error", "transpose"):
        total = _log_int(rng, 1 << 12, 1 << (24 if kind == "squared_error" else 25))
        rows = _log_int(rng, 8, total // 8)
        case["rows"], case["cols"] = rows, max(8, total // rows)
        if kind == "transpose":
            case["dtype"] = rng.choice(["f32", "f32", "f32", "i32"])
    elif kind == "cross_entropy":
        case["batch"], case["classes"] = _log_int(rng, 16, 8192), _log_int(rng, 2, 4000)
    elif kind == "linear":
        case["batch"] = _log_int(rng, 1, 8192)
        case["inputs"], case["outputs"] = _log_int(rng, 64, 4096), _log_int(rng, 10, 4096)
    elif kind == "linear_grad":
        case["batch"] = _log_int(rng, 16, 8192)
        case["inputs"], case["outputs"] = _log_int(rng, 64, 4096), _log_int(rng, 10, 2048)
    elif kind == "train_loop":
        case["batch"], case["steps"] = _log_int(rng, 16, 1024), rng.randint(20, 60)
        case["dims"] = "784,%d,%d" % (_log_int(rng, 32, 512), rng.choice([10, 10, 26]))
    else:
        case["batch"] = _log_int(rng, 64, 8192)
        case["dims"] = "784,%d,%d,10" % (_log_int(rng, 128, 4096), _log_int(rng, 128, 4096))
    return case


# ── inputs, from the seed alone ─────────────────────────────────────────────


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


class _Draws:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def one_hot(self, n, classes):
        labels = torch.randint(classes, (n,), generator=self.g, device="cuda")
        return torch.nn.functional.one_hot(labels, classes).float()

    def integers(self, *shape):
        return torch.randint(-1000, 1000, shape, generator=self.g, device="cuda", dtype=torch.int32)


def _inputs(case, seed):
    d, kind = _Draws(seed), case["kind"]
    if kind == "pointwise":
        return {k: d.uniform(-1, 1, case["n"]) for k in "abc"}
    if kind in ("row_sum", "col_sum"):
        return {"x": d.normal(case["rows"], case["cols"])}
    if kind == "squared_error":
        return {k: d.normal(case["rows"], case["cols"]) for k in ("y", "t")}
    if kind == "transpose":
        shape = (case["rows"], case["cols"])
        return {"x": d.normal(*shape) if case["dtype"] == "f32" else d.integers(*shape)}
    if kind == "cross_entropy":
        return {"z": 3.0 * d.normal(case["batch"], case["classes"]), "t": d.one_hot(case["batch"], case["classes"])}
    if kind in ("linear", "linear_grad"):
        k, n = case["inputs"], case["outputs"]
        got = {"x": d.normal(case["batch"], k), "w0": d.uniform(-1, 1, n, k) / math.sqrt(k),
               "b0": d.uniform(-1, 1, n) / math.sqrt(k)}
        if kind == "linear_grad":
            got["g"] = d.normal(case["batch"], n)
        return got
    dims = _dims(case)
    rows = case["batch"] * (8 if kind == "train_loop" else 1)
    got = {"x": d.uniform(0, 1, rows, dims[0])}
    if kind != "forward":
        got["t"] = d.one_hot(rows, dims[-1])
    for i in range(len(dims) - 1):
        got["w%d" % i] = d.normal(dims[i + 1], dims[i]) * math.sqrt(2.0 / dims[i])
        got["b%d" % i] = d.uniform(-1, 1, dims[i + 1]) / math.sqrt(dims[i])
    return got


def _tensor(x):
    return Tensor.new(x.cpu().numpy(), list(x.shape), "hip")


def _set(p, value):
    p.realize()
    p.write(value.cpu().numpy())


class _Buffer:
    """A realised tensor's device buffer, for torch to view; keeps the tensor."""

    def __init__(self, t):
        self.t = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": "<i4" if t.dtype == fg.I32 else "<f4",
                                         "data": (t.data_ptr()[0], False), "version": 2}


def _view(t):
    return torch.as_tensor(_Buffer(t), device="cuda")


# ── the calls ───────────────────────────────────────────────────────────────


def prepare(case, seed):
    kind = case["kind"]
    data = _inputs(case, seed)
    state = {"kind": kind, "case": case}
    weights = {k: data.pop(k) for k in list(data) if k[0] in "wb" and k[1:].isdigit()}
    for k, v in data.items():
        state[k] = _tensor(v)
    if kind in ("row_sum", "pointwise"):
        state["half"], state["one"] = Tensor.scalar(0.5, "hip"), Tensor.scalar(1.0, "hip")
    if kind in ("linear", "linear_grad"):
        layer = state["layer"] = Linear(case["inputs"], case["outputs"], "hip")
        layers = [layer]
        if kind == "linear_grad":
            state["x"].with_requires_grad(True)
    elif kind in ("forward", "train_loop", "train_step"):
        model = state["model"] = Mlp(_dims(case), "hip")
        layers = model.layers
    else:
        layers = []
        if kind == "cross_entropy":
            state["z"].with_requires_grad(True)
    for i, layer in enumerate(layers):
        _set(layer.weight, weights["w%d" % i])
        _set(layer.bias, weights["b%d" % i])
    if kind in ("train_loop", "train_step"):
        params = model.parameters()
        state["opt"] = Sgd(params, LR)
        state["params"] = [_view(p) for p in params]  # updated in place
    fg.synchronize("hip")
    return state


def run(s):
    kind = s["kind"]
    if kind == "forward":
        return _view(s["model"].forward(s["x"]).realize())
    if kind == "pointwise":
        return _view(s["a"].mul(s["b"]).add(s["c"]).relu().realize())
    if kind == "row_sum":
        return _view(s["x"].mul(s["half"]).add(s["one"]).relu().sum([1]).realize())
    if kind == "col_sum":
        return _view(s["x"].sum([0]).realize())
    if kind == "squared_error":
        d = s["y"].sub(s["t"])
        return _view(d.mul(d).sum([0, 1]).realize())
    if kind == "transpose":
        return _view(s["x"].permute([1, 0]).contiguous().realize())
    if kind == "cross_entropy":
        loss = s["z"].cross_entropy(s["t"])
        grad = loss.gradient([s["z"]])[0]
        Tensor.realize_many([grad, loss])
        return [_view(loss), _view(grad)]
    if kind == "linear":
        return _view(s["layer"](s["x"]).realize())
    if kind == "linear_grad":
        x, layer = s["x"], s["layer"]
        y = layer(x)
        grads = y.mul(s["g"]).sum([0, 1]).gradient([x, layer.weight, layer.bias])
        Tensor.realize_many([y, *grads])
        return [_view(y)] + [_view(g) for g in grads]
    if kind == "train_loop":
        c = s["case"]
        losses = train_batches_native(s["model"], s["opt"], s["x"], s["t"], c["batch"], c["steps"])
        return {"losses": torch.tensor(losses), "params": s["params"]}
    zs = []
    loss = train_step(s["model"], s["opt"], s["x"], s["t"], zs)
    return {"loss": loss.to_vec()[0], "logits": _view(zs[-1]), "params": s["params"]}


# ── what a pass cannot do without ───────────────────────────────────────────


def work(case):
    kind = case["kind"]
    if kind == "pointwise":
        return {"bytes": 16 * case["n"], "flops": 3 * case["n"]}
    if kind in ("row_sum", "col_sum", "squared_error", "transpose"):
        r, c = case["rows"], case["cols"]
        read, wrote, ops = {"row_sum": (1, r, 4), "col_sum": (1, c, 1), "squared_error": (2, 1, 3),
                            "transpose": (1, r * c, 0)}[kind]
        return {"bytes": 4 * (read * r * c + wrote), "flops": ops * r * c}
    if kind == "cross_entropy":
        n = case["batch"] * case["classes"]
        return {"bytes": 4 * (3 * n + 1), "flops": 10 * n}
    if kind in ("linear", "linear_grad"):
        m, k, n = case["batch"], case["inputs"], case["outputs"]
        one = m * k + n * k + n + m * n
        if kind == "linear":
            return {"bytes": 4 * one, "flops": 2 * m * n * k}
        return {"bytes": 4 * (one + m * n + m * k + n * k + n), "flops": 6 * m * n * k}
    dims, b = _dims(case), case["batch"]
    pairs = list(zip(dims, dims[1:]))
    weights = sum(k * n + n for k, n in pairs)
    forward = sum(2 * b * k * n for k, n in pairs)
    if kind == "forward":
        return {"bytes": 4 * (b * dims[0] + weights + b * dims[-1]), "flops": forward}
    step = {"bytes": 4 * (b * (dims[0] + dims[-1]) + 2 * weights), "flops": 3 * forward - 2 * b * dims[0] * dims[1]}
    return {k: v * case.get("steps", 1) for k, v in step.items()}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pointwise", "transpose"):
        return "exact"  # each op rounded once; a copy
    # Four times the errors against exact() that were measured over the ranges
    # of draw(): row and column sums to 1.4e-7 (a column of 60,000), the sum of
    # a whole tensor to 6e-5 (one float32 accumulator over a tall tensor of
    # 2^24 elements), cross-entropy and its gradient to 1.4e-7, products to
    # 1.6e-6 (8192 terms), logits, losses and updated weights to 8.3e-7.
    return {"rel": {"row_sum": 1e-6, "col_sum": 1e-6, "squared_error": 2.5e-4, "cross_entropy": 1e-6,
                    "linear": 6e-6, "linear_grad": 6e-6}.get(kind, 4e-6)}


# ── the same in 64 bits ─────────────────────────────────────────────────────


def _forward64(x, ws, bs):
    pre, h = [], x
    for i, (w, b) in enumerate(zip(ws, bs)):
        z = h @ w.T + b
        pre.append(z)
        h = z.clamp(min=0.0)
    return pre


def _step64(x, t, ws, bs):
    """One SGD step in place; the loss and the logits before it."""
    pre = _forward64(x, ws, bs)
    logp = torch.log_softmax(pre[-1], dim=1)
    loss = -(t * logp).sum() / x.shape[0]
    dz = (logp.exp() * t.sum(1, keepdim=True) - t) / x.shape[0]
    for i in reversed(range(len(ws))):
        h = pre[i - 1].clamp(min=0.0) if i else x
        dw, db = dz.T @ h, dz.sum(0)
        if i:
            dz = (dz @ ws[i]) * (pre[i - 1] > 0)
        ws[i] -= float(torch.tensor(LR)) * dw  # the float32 learning rate
        bs[i] -= float(torch.tensor(LR)) * db
    return loss, pre[-1]


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind in ("pointwise", "transpose"):
        if kind == "transpose":
            return d["x"].T.contiguous()
        # float32 with each op rounded once is the result's definition.
        t = d["a"] * d["b"] + d["c"]
        return torch.where(t > 0, t, torch.zeros_like(t))
    d = {k: v.double() for k, v in d.items()}
    if kind == "row_sum":
        return (d["x"] * 0.5 + 1.0).clamp(min=0.0).sum(1, keepdim=True)
    if kind == "col_sum":
        return d["x"].sum(0, keepdim=True)
    if kind == "squared_error":
        return (d["y"] - d["t"]).square().sum().reshape(1, 1)
    if kind == "cross_entropy":
        logp = torch.log_softmax(d["z"], dim=1)
        n = case["batch"]
        return [-(d["t"] * logp).sum() / n, (logp.exp() - d["t"]) / n]
    if kind in ("linear", "linear_grad"):
        y = d["x"] @ d["w0"].T + d["b0"]
        if kind == "linear":
            return y
        return [y, d["g"] @ d["w0"], d["g"].T @ d["x"], d["g"].sum(0)]
    n = len(_dims(case)) - 1
    ws, bs = [d["w%d" % i] for i in range(n)], [d["b%d" % i] for i in range(n)]
    if kind == "forward":
        return _forward64(d["x"], ws, bs)[-1]
    params = [p for pair in zip(ws, bs) for p in pair]
    if kind == "train_step":
        loss, logits = _step64(d["x"], d["t"], ws, bs)
        return {"loss": loss, "logits": logits, "params": params}
    losses, b = [], case["batch"]
    for i in range(case["steps"]):
        at = (i % 8) * b
        losses.append(_step64(d["x"][at:at + b], d["t"][at:at + b], ws, bs)[0])
    return {"losses": torch.stack(losses), "params": params}
