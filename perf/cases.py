"""Timed workloads of the framework, each one pass through its public entry points.

Every case names its `kind`; the listed cases stand for the work that programs
of this framework do, from the smallest call to the largest, and draw() gives
more cases of the same kinds over the whole range of sizes, layouts and types:

  matmul   one matrix product, or one batch of them (f32, bf16, f64; NN/NT/TN/TT)
  mlp      one SGD step of the two-layer sigmoid network (the fused step)
  tape     one training step written with the reverse-mode tape: two dense
           layers with row biases, tanh, mean squared error, SGD
  layer    a dense layer's row bias and activation, forward and backward
  reduce   the stdlib's Mean, Max and argmax of one array, as host values
  escape   the escape-count map of a grid and the exact sum of its counts

Inputs are made by torch on the GPU from the seed alone and copied into the
library's buffers; outputs come back as torch views of library buffers.
"""
import math

import torch

import cleave_amd as ca
from cleave_amd import autograd

_TYPESTR = {"f32": "<f4", "f64": "<f8", "bf16": "<i2", "u32": "<i4", "u64": "<i8", "i64": "<i8"}
_TORCH = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f64": 8, "bf16": 2}
_LR = 0.01


def listed():
    return [
        # the smallest product, bound by its launch: one call of a program that works on small tensors
        {"name": "f32_256", "kind": "matmul", "dtype": "f32", "batch": 1, "m": 256, "n": 256, "k": 256,
         "ta": False, "tb": False},
        # the large f32 product, the benchmark's headline
        {"name": "f32_4096", "kind": "matmul", "dtype": "f32", "batch": 1, "m": 4096, "n": 4096, "k": 4096,
         "ta": False, "tb": False},
        # the weight gradient X^T g of a ragged layer over a batch of 10000 rows
        {"name": "f32_weight_grad", "kind": "matmul", "dtype": "f32", "batch": 1, "m": 784, "n": 500, "k": 10000,
         "ta": True, "tb": False},
        # the large bf16 product of the benchmark, the largest by operations
        {"name": "bf16_8192", "kind": "matmul", "dtype": "bf16", "batch": 1, "m": 8192, "n": 8192, "k": 8192,
         "ta": False, "tb": False},
        # the benchmark's batch of small bf16 products
        {"name": "bf16_batched", "kind": "matmul", "dtype": "bf16", "batch": 64, "m": 512, "n": 512, "k": 512,
         "ta": False, "tb": False},
        # Tensor<f64>: an ordinary product that does not fill whole tiles
        {"name": "f64_1000", "kind": "matmul", "dtype": "f64", "batch": 1, "m": 1000, "n": 1000, "k": 1000,
         "ta": False, "tb": False},
        # the benchmark's training step, the largest by time
        {"name": "mlp_large", "kind": "mlp", "b": 65536, "d": 1024, "h": 4096},
        # the same step on an ordinary ragged network and minibatch
        {"name": "mlp_minibatch", "kind": "mlp", "b": 1000, "d": 784, "h": 300},
        # a classifier's training step written by its user on the tape: 10 outputs
        {"name": "tape_classifier", "kind": "tape", "b": 4096, "d": 784, "h": 256, "c": 10},
        # bias, tanh and their backward over a large batch of a wide layer
        {"name": "layer_tanh", "kind": "layer", "dtype": "f32", "rows": 20000, "cols": 1000, "act": "tanh"},
        # losses of a data set reduced to the numbers a program prints
        {"name": "reduce_10m", "kind": "reduce", "dtype": "f32", "n": 10_000_000},
        # the benchmark's escape-count grid over the whole set
        {"name": "escape_16384", "kind": "escape", "width": 16384, "height": 16384, "x0": -2.0, "y0": -1.5,
         "span": 3.0, "max_iter": 1000},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]: half of them multiples of 8 or 64, half as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    q = rng.choice((1, 1, 8, 64))
    return max(lo, min(hi, (v + q - 1) // q * q if q > 1 else v))


def draw(rng):
    kind = rng.choice(("matmul", "matmul", "matmul", "mlp", "tape", "layer", "reduce", "escape"))
    if kind == "matmul":
        dtype = rng.choice(("f32", "f32", "bf16", "f64"))
        most = 2.0 * 8192**3 if dtype == "bf16" else 2.0 * 4096**3
        batch = rng.choice((1, 1, 1, 0))
        batch = batch or rng.randint(2, 64)
        while True:
            m, k = _size(rng, 32, 8192), _size(rng, 32, 16384)
            # one product in six has a narrow operand: a column, or a head of a few classes
            n = rng.choice((1, 2, 10, 16)) if rng.randrange(6) == 0 else _size(rng, 32, 8192)
            if 2.0 * batch * m * n * k <= most and batch * max(m * n, m * k, n * k) <= 1 << 27:
                break
        return {"kind": kind, "dtype": dtype, "batch": batch, "m": m, "n": n, "k": k,
                "ta": bool(rng.randrange(2)), "tb": bool(rng.randrange(2))}
    if kind == "mlp":
        return {"kind": kind, "b": _size(rng, 64, 32768), "d": _size(rng, 8, 1024), "h": _size(rng, 8, 2048)}
    if kind == "tape":
        return {"kind": kind, "b": _size(rng, 64, 8192), "d": _size(rng, 8, 1024), "h": _size(rng, 16, 1024),
                "c": rng.randint(2, 100)}
    if kind == "layer":
        while True:
            rows, cols = _size(rng, 64, 20000), _size(rng, 8, 8192)
            if rows * cols <= 1 << 26:
                break
        return {"kind": kind, "dtype": rng.choice(("f32", "f32", "f64")), "rows": rows, "cols": cols,
                "act": rng.choice(("tanh", "sigmoid", "relu"))}
    if kind == "reduce":
        return {"kind": kind, "dtype": rng.choice(("f32", "f32", "f64")), "n": _size(rng, 1000, 1 << 27)}
    # a window on the set: the whole of it down to one 200th, so that its edge fills the grid
    span = 3.0 * math.exp(-rng.uniform(0.0, math.log(200.0)))
    cx, cy = rng.choice(((-0.5, 0.0), (-0.75, 0.1), (-1.25, 0.0), (-0.16, 1.03), (0.28, 0.01)))
    return {"kind": kind, "width": _size(rng, 256, 8192), "height": _size(rng, 256, 8192),
            "x0": round(cx - span / 2, 6), "y0": round(cy - span / 2, 6), "span": round(span, 6),
            "max_iter": _size(rng, 50, 1000)}


# ---- inputs ----------------------------------------------------------------------


def _inputs(case, seed):
    """The case's operands as torch tensors on the GPU, in the dtype that the call takes."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(shape, dtype="f32", std=1.0):
        # bf16 and f64 operands are draws of their own width, rounded once
        t = torch.randn(shape, device="cuda", generator=g, dtype=torch.float64 if dtype == "f64" else torch.float32)
        return t.mul_(std).to(_TORCH[dtype])

    def uniform(shape, lim):
        return torch.rand(shape, device="cuda", generator=g).mul_(2 * lim).sub_(lim)

    kind = case["kind"]
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        std = 0.02 if dt == "bf16" else 1.0
        return {"a": normal(lead + ((k, m) if case["ta"] else (m, k)), dt, std),
                "b": normal(lead + ((n, k) if case["tb"] else (k, n)), dt, std)}
    if kind == "mlp":  # N(0,1) features, targets in {0,1}, Xavier-uniform weights
        b, d, h = case["b"], case["d"], case["h"]
        return {"x": normal((b, d)), "y": (torch.rand(b, device="cuda", generator=g) < 0.5).float(),
                "w1": uniform((d, h), math.sqrt(6.0 / (d + h))), "w2": uniform((h,), math.sqrt(6.0 / (h + 1)))}
    if kind == "tape":
        b, d, h, c = case["b"], case["d"], case["h"], case["c"]
        cls = torch.randint(0, c, (b,), device="cuda", generator=g)
        return {"x": normal((b, d)), "y": torch.nn.functional.one_hot(cls, c).float(),
                "w1": uniform((d, h), math.sqrt(6.0 / (d + h))), "b1": uniform((h,), 0.1),
                "w2": uniform((h, c), math.sqrt(6.0 / (h + c))), "b2": uniform((c,), 0.1)}
    if kind == "layer":
        shape, dt = (case["rows"], case["cols"]), case["dtype"]
        return {"a": normal(shape, dt), "bias": normal((case["cols"],), dt, 0.1), "g": normal(shape, dt, 0.01)}
    if kind == "reduce":  # losses: none is negative
        return {"x": normal((case["n"],), case["dtype"]).abs_()}
    return {"shift": torch.rand(2, generator=torch.Generator().manual_seed(seed))}  # escape: where the grid starts


class _Buffer:
    """The array interface of a library tensor, for torch views of its memory; keeps the tensor alive."""

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": _TYPESTR[t.dtype],
                                         "data": (t.ptr, False), "version": 2}


def _view(t):
    return torch.as_tensor(_Buffer(t), device="cuda")


def _upload(x):
    """A library tensor with the values of the torch tensor x."""
    dtype = {torch.float32: "f32", torch.float64: "f64", torch.bfloat16: "bf16"}[x.dtype]
    t = ca.empty(tuple(x.shape), dtype)
    _view(t).copy_(x.view(torch.int16) if dtype == "bf16" else x)
    return t


def prepare(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    s = {"case": case}
    if kind == "escape":
        w, h = case["width"], case["height"]
        step = case["span"] / max(w, h)
        # grids of other seeds start up to half a pixel away
        s["grid"] = (w, h, case["x0"] + 0.5 * step * float(x["shift"][0]),
                     case["y0"] + 0.5 * step * float(x["shift"][1]), step, step, case["max_iter"])
        s["counts"], s["total"] = ca.empty((h, w), "u32"), ca.empty((1,), "u64")
        s["out"] = {"counts": _view(s["counts"]), "total": _view(s["total"])}
        return s
    for name, v in x.items():
        s[name] = _upload(v)
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        s["c"] = ca.empty(lead + (case["m"], case["n"]), "f64" if case["dtype"] == "f64" else "f32")
        s["out"] = _view(s["c"])
    elif kind == "mlp":
        s["dw1"], s["dw2"], s["loss"] = ca.empty((case["d"], case["h"])), ca.empty((case["h"],)), ca.empty((1,))
        s["out"] = {n: _view(s[n]) for n in ("dw1", "dw2", "loss", "w1", "w2")}
    elif kind == "layer":
        shape, dt = (case["rows"], case["cols"]), case["dtype"]
        for n in ("z", "t", "dz"):
            s[n] = ca.empty(shape, dt)
        s["db"] = ca.empty((case["cols"],), dt)
        s["out"] = {n: _view(s[n]) for n in ("z", "t", "dz", "db")}
    torch.cuda.synchronize()  # the copies above ran on torch's stream, the library has its own
    return s


# ---- one pass --------------------------------------------------------------------


def _tape_step(s):
    """Forward, backward and SGD update of tanh(x w1 + b1) w2 + b2 under the mean squared error."""
    x, y = autograd.const(s["x"]), autograd.const(s["y"])
    w1, b1, w2, b2 = (autograd.param(s[n]) for n in ("w1", "b1", "w2", "b2"))
    hidden = autograd.tanh(autograd.add_row_bias(x @ w1, b1))
    e = autograd.add_row_bias(hidden @ w2, b2) - y
    loss = autograd.mean(e * e)
    autograd.backward(loss)
    out = {"loss": loss.tensor}
    for n, p in (("w1", w1), ("b1", b1), ("w2", w2), ("b2", b2)):
        ca.sgd_update(p.tensor, p.grad, _LR)
        out[n] = p.grad
    return {n: _view(t) for n, t in out.items()}


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "matmul":
        if case["batch"] > 1:
            ca.matmul_batched(s["a"], s["b"], out=s["c"], trans_a=case["ta"], trans_b=case["tb"])
        else:
            ca.matmul(s["a"], s["b"], trans_a=case["ta"], trans_b=case["tb"], out=s["c"])
    elif kind == "mlp":
        ca.mlp_step(s["x"], s["y"], s["w1"], s["w2"], _LR, dw1=s["dw1"], dw2=s["dw2"], loss=s["loss"])
    elif kind == "tape":
        return _tape_step(s)
    elif kind == "layer":
        ca.add_row_bias(s["a"], s["bias"], out=s["z"])
        if case["act"] == "tanh":
            ca.tanh(s["z"], out=s["t"])
            ca.tanh_bwd(s["t"], s["g"], out=s["dz"])
        elif case["act"] == "sigmoid":
            ca.sigmoid(s["z"], out=s["t"])
            ca.sigmoid_bwd(s["t"], s["g"], out=s["dz"])
        else:
            ca.relu(s["z"], out=s["t"])
            ca.relu_bwd(s["z"], s["g"], out=s["dz"])
        ca.sum_rows(s["dz"], out=s["db"])
    elif kind == "reduce":
        return {"mean": ca.mean(s["x"]), "max": ca.max_of(s["x"]), "argmax": ca.argmax(s["x"])}
    else:
        ca.escape_counts(*s["grid"], out=s["counts"])
        ca.reduce_sum_u64(s["counts"], s["total"])
    return s["out"]


# ---- what a pass cannot do without, and what it must give ------------------------


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        batch, m, n, k, e = case["batch"], case["m"], case["n"], case["k"], _SIZE[case["dtype"]]
        return {"bytes": batch * ((m * k + k * n) * e + m * n * max(e, 4)), "flops": 2.0 * batch * m * n * k}
    if kind == "mlp":
        # x read; w1, w2 read and written; dw1, dw2 written; x w1 and x^T d1, and the products with w2
        b, d, h = case["b"], case["d"], case["h"]
        return {"bytes": 4 * (b * d + b + 3 * d * h + 3 * h + 1), "flops": 4.0 * b * d * h + 4.0 * b * h}
    if kind == "tape":
        b, d, h, c = case["b"], case["d"], case["h"], case["c"]
        p = d * h + h + h * c + c
        return {"bytes": 4 * (b * d + b * c + 3 * p + 1), "flops": 4.0 * b * d * h + 6.0 * b * h * c}
    if kind == "layer":
        n, e = case["rows"] * case["cols"], _SIZE[case["dtype"]]
        return {"bytes": e * (5 * n + 2 * case["cols"]), "flops": 8.0 * n}
    if kind == "reduce":
        return {"bytes": case["n"] * _SIZE[case["dtype"]], "flops": 3.0 * case["n"]}
    n = case["width"] * case["height"]
    return {"bytes": 4.0 * n, "flops": 11.0 * n}  # every count written, at least one iteration each


def tolerance(case):
    if case["kind"] == "escape":
        return "exact"
    if case.get("dtype") == "f64":
        return {"rel": 2e-14}
    # sums of f32 products; the gradients of a step carry the rounding of two or three such sums
    return {"rel": 1e-5}


def exact(case, seed):
    kind = case["kind"]
    if kind == "escape":
        return None  # whole numbers, defined by their f32 arithmetic
    x = {n: v.double() for n, v in _inputs(case, seed).items()}
    if kind == "matmul":
        a = x["a"].transpose(-1, -2).contiguous() if case["ta"] else x["a"]
        b = x["b"].transpose(-1, -2).contiguous() if case["tb"] else x["b"]
        return a @ b
    if kind == "mlp":
        hid = torch.sigmoid(x["x"] @ x["w1"])
        yh = torch.sigmoid(hid @ x["w2"])
        e = yh - x["y"]
        d2 = 2.0 * e / case["b"] * yh * (1.0 - yh)
        dw2 = hid.t() @ d2
        d1 = d2[:, None] * x["w2"][None, :] * hid * (1.0 - hid)
        dw1 = x["x"].t() @ d1
        return {"dw1": dw1, "dw2": dw2, "loss": (e * e).mean().reshape(1), "w1": x["w1"] - _LR * dw1,
                "w2": x["w2"] - _LR * dw2}
    if kind == "tape":
        hid = torch.tanh(x["x"] @ x["w1"] + x["b1"])
        e = hid @ x["w2"] + x["b2"] - x["y"]
        go = 2.0 * e / e.numel()
        gz = (go @ x["w2"].t()) * (1.0 - hid * hid)
        return {"loss": (e * e).mean().reshape(1), "w1": x["x"].t() @ gz, "b1": gz.sum(0),
                "w2": hid.t() @ go, "b2": go.sum(0)}
    if kind == "layer":
        z = x["a"] + x["bias"]
        if case["act"] == "tanh":
            t = torch.tanh(z)
            dz = x["g"] * (1.0 - t * t)
        elif case["act"] == "sigmoid":
            t = torch.sigmoid(z)
            dz = x["g"] * t * (1.0 - t)
        else:
            t = torch.relu(z)
            dz = torch.where(z > 0, x["g"], torch.zeros_like(z))
        return {"z": z, "t": t, "dz": dz, "db": dz.sum(0)}
    return {"mean": float(x["x"].mean()), "max": float(x["x"].max()), "argmax": int(x["x"].argmax())}
