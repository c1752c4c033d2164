"""The work that is measured: what programs written against this library have it do, through its public entry points.

A case is a dict of plain values; its "kind" names the program.  Sizes are those of this repository's benchmark and tests or generic ones:

* ``mlp``      one training step of a multi-layer perceptron: ``diff`` of ``nll(predict(x), labels)`` and ``update_`` of every parameter.
               ``layers`` is how the program writes its layers: "plain" (``relu(w @ x + b)``, as the reference's examples do) or "dense" (the README's).
* ``words``    one training step of a word model: embedding lookup of a batch of words, a hidden layer, scores over the whole vocabulary, ``nll``
               of the next word.  Words are drawn by Zipf's law, as in text.
* ``actback``  the gradient of an activation function on its own.
* ``unbroadcast``  the gradient of a bias: ``sum(dy; dims)``, of a dense layer (2 dims) or of a convolution layer (4 dims).
* ``xent``     value and gradient of ``nll`` on a matrix of scores that is there already.
* ``softmax``  ``softmax`` / ``logsoftmax`` and its gradient down any one dimension.
* ``stats``    ``mean`` and ``var`` as normalisation layers take them.

Arrays belong to the program (torch tensors that ``KnetArray.from_torch`` wraps); results that the library allocates are handed over without a copy.
"""
import math

import numpy as np
import torch

import __graft_entry__

K = __graft_entry__.load_package()

TYPES = {"f32": torch.float32, "f64": torch.float64}
SIZE = {"f32": 4, "f64": 8}
ACTS = ("relu", "sigm", "tanh", "elu", "selu")


def listed():
    return [
        # the tutorial's model at its batch size: every call is small, so what counts is the number of launches and the host's share of each
        {"name": "mlp_784_64_10", "kind": "mlp", "input": 784, "width": 64, "hidden": 1, "classes": 10, "batch": 100, "layers": "plain",
         "pdrop": 0.0, "fused": False, "opt": "adam", "type": "f32"},
        # an ordinary model written with the README's layers; odd batch (the last one of an epoch)
        {"name": "mlp_784_1000x2_b237", "kind": "mlp", "input": 784, "width": 1000, "hidden": 2, "classes": 100, "batch": 237, "layers": "dense",
         "pdrop": 0.0, "fused": False, "opt": "adam", "type": "f32"},
        # the benchmark's deep model: 7 hidden layers of 4096, relu and dropout, 1000 classes, batch 2048
        {"name": "mlp_4096x7_drop", "kind": "mlp", "input": 4096, "width": 4096, "hidden": 7, "classes": 1000, "batch": 2048, "layers": "plain",
         "pdrop": 0.5, "fused": True, "opt": "momentum", "type": "f32"},
        # vocabulary and width of the embedding tests, 2048 words a step
        {"name": "words_32000x512_b2048", "kind": "words", "vocab": 32000, "width": 512, "batch": 2048, "opt": "adam", "type": "f32"},
        # the benchmark's isolated gradients: one of the five, at full size
        {"name": "tanhback_2e28", "kind": "actback", "act": "tanh", "n": 1 << 28, "type": "f32"},
        # bias gradient of the small model's hidden layer: one launch, all latency
        {"name": "bias_64x100", "kind": "unbroadcast", "dims": "64,100", "over": "2", "type": "f32"},
        # the benchmark's reductions: a wide dense layer, and a convolution layer
        {"name": "bias_4096x8192", "kind": "unbroadcast", "dims": "4096,8192", "over": "2", "type": "f32"},
        {"name": "convbias_56_256_64", "kind": "unbroadcast", "dims": "56,56,256,64", "over": "1,2,4", "type": "f32"},
        # the benchmark's losses: a vocabulary through nll as it is called by default, and the small one in doubles through the one-pass form
        {"name": "xent_32000x512", "kind": "xent", "classes": 32000, "batch": 512, "fused": False, "type": "f32"},
        {"name": "xent_1000x4096_f64", "kind": "xent", "classes": 1000, "batch": 4096, "fused": True, "type": "f64"},
        # the shape the reference's own softmax measurements are quoted at
        {"name": "logsoftmax_100000x100", "kind": "softmax", "op": "logsoftmax", "dims": "100000,100", "over": 1, "type": "f32"},
        # statistics of a convolution layer's output, odd sizes
        {"name": "stats_29_193_64", "kind": "stats", "dims": "29,29,193,64", "over": "1,2,4", "type": "f32"},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _type(rng):
    return "f64" if rng.random() < 0.25 else "f32"


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "words", "actback", "unbroadcast", "unbroadcast", "xent", "xent", "softmax", "softmax", "stats"])
    if kind == "mlp":
        width = _log(rng, 32, 3500)
        layers = rng.choice(["plain", "dense"])
        return {"kind": kind, "input": _log(rng, 64, 4096), "width": width, "hidden": rng.randint(1, 6), "classes": _log(rng, 10, 1000),
                "batch": _log(rng, 16, 2048), "layers": layers, "pdrop": rng.choice([0.0, 0.2, 0.5]) if layers == "plain" else 0.0,
                "fused": rng.random() < 0.3, "opt": rng.choice(["sgd", "momentum", "adam"]), "type": "f64" if width <= 512 and rng.random() < 0.2 else "f32"}
    if kind == "words":
        vocab = _log(rng, 1000, 32000)
        return {"kind": kind, "vocab": vocab, "width": _log(rng, 64, 512), "batch": _log(rng, 64, 2048), "opt": rng.choice(["sgd", "adam"]), "type": "f32"}
    t = _type(rng)
    half = 1 if t == "f32" else 2
    if kind == "actback":
        return {"kind": kind, "act": rng.choice(ACTS), "n": _log(rng, 1000, (1 << 28) // half), "type": t}
    if kind == "unbroadcast":
        if rng.random() < 0.4:
            side, channels = rng.randint(5, 64), _log(rng, 16, 1024)
            batch = max(2, min(_log(rng, 8, 256), 40_000_000 // half // (side * side * channels)))
            return {"kind": kind, "dims": "%d,%d,%d,%d" % (side, side, channels, batch), "over": "1,2,4", "type": t}
        rows = _log(rng, 10, 32000)
        return {"kind": kind, "dims": "%d,%d" % (rows, _log(rng, 16, max(17, min(50000, 40_000_000 // half // rows)))), "over": rng.choice(["1", "2"]), "type": t}
    if kind == "xent":
        classes = _log(rng, 2, 50000)
        return {"kind": kind, "classes": classes, "batch": _log(rng, 16, max(17, min(100_000, 25_000_000 // half // classes))), "fused": rng.random() < 0.5, "type": t}
    if kind == "softmax":
        op = rng.choice(["softmax", "logsoftmax"])
        if rng.random() < 0.5:
            rows = _log(rng, 10, 100_000)
            return {"kind": kind, "op": op, "dims": "%d,%d" % (rows, _log(rng, 16, max(17, min(100_000, 20_000_000 // half // rows)))), "over": rng.choice([1, 1, 2]), "type": t}
        a, b = _log(rng, 8, 256), _log(rng, 8, 1024)
        return {"kind": kind, "op": op, "dims": "%d,%d,%d" % (a, b, max(2, _log(rng, 4, max(5, 20_000_000 // half // (a * b))))), "over": rng.choice([1, 2]), "type": t}
    if rng.random() < 0.5:
        side, channels = rng.randint(5, 57), _log(rng, 16, 512)
        batch = max(2, min(_log(rng, 8, 128), 25_000_000 // half // (side * side * channels)))
        return {"kind": "stats", "dims": "%d,%d,%d,%d" % (side, side, channels, batch), "over": "1,2,4", "type": t}
    rows = _log(rng, 32, 8192)
    return {"kind": "stats", "dims": "%d,%d" % (rows, _log(rng, 32, min(50000, 25_000_000 // half // rows))), "over": rng.choice(["1", "2"]), "type": t}


# ---- what a program has in hand -------------------------------------------------------------------------------------------------------

def _ints(text):
    return [int(v) for v in text.split(",")]


class _Given:
    """Hands an array that the library allocated to torch, without a copy; the memory goes back to the library with the last tensor on it."""

    def __init__(self, a):
        self.a = a
        strides, s = [], a.dtype.itemsize
        for d in a.dims:
            strides.append(s)
            s *= d
        self.__cuda_array_interface__ = {"shape": tuple(a.dims), "strides": tuple(strides), "typestr": a.dtype.str, "data": (a.ptr, False), "version": 2}


def _torch(a):
    return torch.as_tensor(_Given(a), device="cuda")


def _normal(gen, n, dtype, scale=1.0):
    """n draws of N(0, scale^2): made in doubles, so that both types hold the same numbers."""
    out = torch.empty(n, dtype=dtype, device="cuda")
    for i in range(0, n, 1 << 26):
        part = out[i:i + (1 << 26)]
        part.copy_(torch.randn(part.numel(), dtype=torch.float64, device="cuda", generator=gen).mul_(scale))
    return out


def _wrap(t, *dims):
    return K.KnetArray.from_torch(t, dims=dims)


def _optimizer(case, n, dtype, kept):
    """The optimizer of one parameter and its state, as a program that saves checkpoints holds it."""
    def state():
        kept.append(torch.zeros(n, dtype=dtype, device="cuda"))
        return _wrap(kept[-1], n)
    if case["opt"] == "sgd":
        return K.SGD(lr=0.01)
    if case["opt"] == "momentum":
        o = K.Momentum(lr=0.001, gamma=0.9)
        o.velocity = state()
        return o
    o = K.Adam(lr=0.0001)
    o.fstm, o.scndm = state(), state()
    return o


def _parameters(case, shapes, gen, dtype):
    """(parameters, the tensors behind them and behind their optimizers): weights by fan-in, biases small."""
    params, kept = [], []
    for rows, cols in shapes:
        t = _normal(gen, rows * cols, dtype, math.sqrt(2.0 / cols) if cols > 1 else 0.01)
        kept.append(t)
        p = K.Param(_wrap(t, rows, cols))
        p.opt = _optimizer(case, rows * cols, dtype, kept)
        params.append(p)
    return params, kept


def _mlp_shapes(case):
    sizes = [case["input"]] + [case["width"]] * case["hidden"] + [case["classes"]]
    return [s for i in range(len(sizes) - 1) for s in ((sizes[i + 1], sizes[i]), (sizes[i + 1], 1))]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = np.random.default_rng(seed)
    dtype, kind = TYPES[case["type"]], case["kind"]
    s = {"case": case}
    if kind == "mlp":
        s["params"], s["kept"] = _parameters(case, _mlp_shapes(case), gen, dtype)
        x = torch.rand(case["input"] * case["batch"], dtype=torch.float64, device="cuda", generator=gen).to(dtype)
        s["x"] = _wrap(x, case["input"], case["batch"])
        s["labels"] = host.integers(1, case["classes"] + 1, size=case["batch"])
        K.seed_(seed)                                        # dropout draws from the library's generator
    elif kind == "words":
        v, w, b = case["vocab"], case["width"], case["batch"]
        s["params"], s["kept"] = _parameters(case, [(w, v), (w, w), (w, 1), (v, w), (v, 1)], gen, dtype)
        p = 1.0 / np.arange(1, v + 1)
        order = host.permutation(v) + 1                      # word numbers are not sorted by frequency
        text = order[np.searchsorted(np.cumsum(p / p.sum())[:-1], host.random(b + 1))]
        s["words"], s["labels"] = text[:-1].copy(), text[1:].copy()
    elif kind == "actback":
        x = _wrap(_normal(gen, case["n"], dtype), case["n"])
        s["y"] = getattr(K, case["act"])(x)
        s["dy"] = _wrap(_normal(gen, case["n"], dtype), case["n"])
    else:
        dims = [case["classes"], case["batch"]] if kind == "xent" else _ints(case["dims"])
        x = _wrap(_normal(gen, math.prod(dims), dtype, 2.0 if kind == "xent" else 1.0), *dims)
        if kind == "xent":
            s["scores"] = K.Param(x)
            s["labels"] = host.integers(1, case["classes"] + 1, size=case["batch"])
        else:
            s["x"] = x
        if kind == "softmax":
            s["dy"] = _wrap(_normal(gen, math.prod(dims), dtype), *dims)
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------------------------

def _predict(case, w, h):
    last = len(w) - 2
    for i in range(0, len(w), 2):
        if case["layers"] == "dense":
            h = K.dense(w[i], h, w[i + 1], act="relu" if i < last else None)
            continue
        h = w[i] @ h + w[i + 1]
        if i < last:
            h = K.relu(h)
            if case["pdrop"] > 0:
                h = K.dropout(h, case["pdrop"])
    return h


def _train(s, loss):
    J = K.diff(loss)
    for p in s["params"]:
        K.update_(p, K.grad(J, p))
    return [float(K.value(J))] + s["kept"]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mlp":
        return _train(s, lambda: K.nll(_predict(case, s["params"], s["x"]), s["labels"], fused=case["fused"]))
    if kind == "words":
        we, w1, b1, w2, b2 = s["params"]
        return _train(s, lambda: K.nll(K.dense(w2, K.relu(w1 @ K.getcols(we, s["words"]) + b1), b2), s["labels"]))
    if kind == "actback":
        return _torch(getattr(K, case["act"] + "back")(s["dy"], s["y"]))
    if kind == "unbroadcast":
        return _torch(K.sum(s["x"], dims=_ints(case["over"])))
    if kind == "xent":
        J = K.diff(lambda: K.nll(s["scores"], s["labels"], fused=case["fused"]))
        return float(K.value(J)), _torch(K.grad(J, s["scores"]))
    if kind == "softmax":
        x, dy, op = s["x"], s["dy"], getattr(K, case["op"])
        if case["over"] == 1:
            # forward and backward as a program that has the gradient of the result in hand writes them
            y = op(x, dims=1)
            return _torch(y), _torch(getattr(K, case["op"] + "back")(y, dy, dims=1))
        # along another dimension the gradient is the tape's; its scalar is a sum of terms of both signs, so not an output of its own
        kept, p = [], K.Param(x)

        def scalar():
            y = op(p, dims=case["over"])
            kept.append(K.value(y))
            return K.sum(y * dy)
        J = K.diff(scalar)
        return _torch(kept[0]), _torch(K.grad(J, p))
    m = K.mean(s["x"], dims=_ints(case["over"]))
    return _torch(m), _torch(K.var(s["x"], dims=_ints(case["over"]), mean=m, corrected=False))


# ---- the same in 64 bits, by torch alone ----------------------------------------------------------------------------------------------

def _updated(case, w, g, states):
    """One parameter and its optimizer's state after the first step."""
    if case["opt"] == "sgd":
        return [w - 0.01 * g]
    if case["opt"] == "momentum":
        v = 0.9 * states[0] - 0.001 * g
        return [w + v, v]
    m, v = 0.9 * states[0] + 0.1 * g, 0.999 * states[1] + 0.001 * g * g
    return [w - 0.0001 * (m / 0.1) / (torch.sqrt(v / 0.001) + 1e-8), m, v]


def exact(case, seed):
    """What run returns for these inputs; None where dropout draws from the library's own generator."""
    kind = case["kind"]
    if kind == "mlp" and case["pdrop"] > 0:
        return None
    s = prepare(case, seed)
    torch.cuda.synchronize()

    def double(a):
        return _torch(K.value(a)).double()

    if kind in ("mlp", "words"):
        w = [double(p).requires_grad_() for p in s["params"]]
        if kind == "mlp":
            h = double(s["x"])
            for i in range(0, len(w), 2):
                h = w[i] @ h + w[i + 1]
                h = torch.relu(h) if i < len(w) - 2 else h
        else:
            we, w1, b1, w2, b2 = w
            h = w2 @ torch.relu(w1 @ we[:, torch.as_tensor(s["words"] - 1, device="cuda")] + b1) + b2
        loss = torch.nn.functional.cross_entropy(h.t(), torch.as_tensor(s["labels"] - 1, device="cuda"))
        grads = torch.autograd.grad(loss, w)
        out, each = [loss.item()], len(s["kept"]) // len(w)
        for i, (a, g) in enumerate(zip(w, grads)):
            states = [t.double() for t in s["kept"][i * each + 1:(i + 1) * each]]
            out += _updated(case, a.detach().t().reshape(-1), g.t().reshape(-1), states)
        return out
    if kind == "actback":
        y, dy, act = double(s["y"]), double(s["dy"]), case["act"]
        if act == "relu":
            return dy * (y > 0)
        if act == "sigm":
            return dy * y * (1 - y)
        if act == "tanh":
            return dy * (1 - y) * (1 + y)
        if act == "elu":
            return torch.where(y >= 0, dy, dy * (1 + y))
        scale, alpha = 1.0507009873554805, 1.6732632423543772
        return torch.where(y >= 0, scale * dy, dy * (y + scale * alpha))
    if kind == "xent":
        x = double(s["scores"]).requires_grad_()
        loss = torch.nn.functional.cross_entropy(x.t(), torch.as_tensor(s["labels"] - 1, device="cuda"))
        return loss.item(), torch.autograd.grad(loss, x)[0]
    x = double(s["x"])
    over = [d - 1 for d in (_ints(case["over"]) if kind != "softmax" else [case["over"]])]
    if kind == "unbroadcast":
        return x.sum(over, keepdim=True)
    if kind == "softmax":
        x.requires_grad_()
        y = torch.softmax(x, over[0]) if case["op"] == "softmax" else torch.log_softmax(x, over[0])
        return y.detach(), torch.autograd.grad(y, x, double(s["dy"]))[0]
    return x.mean(over, keepdim=True), x.var(over, correction=0, keepdim=True)


# ---- what a pass cannot do without, and how far another correct implementation may be off ------------------------------------------------

_STATE = {"sgd": 3, "momentum": 5, "adam": 7}                # arrays read or written by an update: gradient, weights twice, state twice each


def work(case):
    size, kind = SIZE[case["type"]], case["kind"]
    if kind == "mlp":
        shapes, b = _mlp_shapes(case), case["batch"]
        weights = sum(r * c for r, c in shapes)
        products = sum(2.0 * r * c * b for r, c in shapes[::2])
        first = 2.0 * shapes[0][0] * shapes[0][1] * b        # the data needs no gradient
        return {"bytes": size * (_STATE[case["opt"]] * weights + case["input"] * b), "flops": 3 * products - first}
    if kind == "words":
        v, w, b = case["vocab"], case["width"], case["batch"]
        weights = 2 * w * v + w * w + w + v
        return {"bytes": size * _STATE[case["opt"]] * weights, "flops": 3 * (2.0 * w * w * b + 2.0 * v * w * b)}
    if kind == "actback":
        return {"bytes": 3 * size * case["n"], "flops": 0}
    if kind == "xent":
        return {"bytes": size * 2 * case["classes"] * case["batch"] + 4 * case["batch"], "flops": 0}
    dims = _ints(case["dims"])
    n = math.prod(dims)
    if kind == "softmax":
        return {"bytes": 4 * size * n, "flops": 0}
    kept = n // math.prod(dims[d - 1] for d in _ints(case["over"]))
    return {"bytes": size * (n + (2 if kind == "stats" else 1) * kept), "flops": 0}


# Measured: each kind run in floats against the same numbers run in doubles (listed and drawn cases; 2-norm of the difference / largest
# difference), then four times the worst:
#   mlp, words   1.4e-3 / 0.19: not rounding as such, which leaves 1e-7 .. 3e-6 here, but the few units whose sum before relu lies within
#                rounding of zero and which one order of summation switches on and another off, each with its share of every gradient before it
#   actback      6.0e-8 / 6.0e-7          unbroadcast  2.0e-7 / 7.4e-7          xent  5.9e-8 / 1.2e-6
#   softmax      9.5e-8 / 9.0e-7          stats        2.1e-7 / 7.4e-7
# Doubles have 29 bits more; exp and log of different libraries differ in their last bit there, and a unit on the edge of relu is too rare to meet.
_TOLERANCE = {"mlp": (5e-3, 0.8), "words": (5e-3, 0.8), "actback": (2.5e-7, 2.5e-6), "unbroadcast": (8e-7, 3e-6), "xent": (2.5e-7, 5e-6),
              "softmax": (4e-7, 4e-6), "stats": (8e-7, 3e-6)}


def tolerance(case):
    rel, most = _TOLERANCE[case["kind"]]
    if case["type"] == "f64":
        rel, most = (1e-11, 1e-9) if case["kind"] in ("mlp", "words") else (1e-14, 1e-13)
    return {"rel": rel, "max": most}
