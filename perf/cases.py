"""The work that is timed: what a program built on this package asks of it between its matrix products.

Tensors belong to torch here and are handed over as `Matrix` views of the same memory; every call goes
through the public surface (the `Matrix` methods, the module's functions and optimizers, and the C entry
points of `zenu_amd.lib()` where the method would allocate its result).  A case is a dict of plain values:

  predict   forward pass of a two-hidden-layer classifier: bias + ReLU twice, bias, softmax, arg-max
  train     the same classifier's training step: forward, cross-entropy, backward with bias gradients,
            the materialised transposes around its matrix products, one AdamW update
  act       an activation and its backward pass over a flat tensor
  bcast     matrix with a row, a column, a transposed matrix and a scalar
  stats     column sums, row sums, row maxima with their positions, sum of magnitudes
  softmax   softmax along one axis of [outer, classes, inner] and its backward pass
  conv      what surrounds a convolution: channel bias, ReLU, both backward, NCHW -> NHWC
  adamw     one optimizer step over the tensors of a model
"""
import ctypes as C
import math

import numpy as np
import torch

import zenu_amd as zenu
from zenu_amd import Matrix, _lib

_TORCH = {"f32": torch.float32, "f64": torch.float64}
_CODE = {"f32": _lib.F32, "f64": _lib.F64}
_SIZE = {"f32": 4, "f64": 8}
_NUMPY = {torch.float32: np.float32, torch.float64: np.float64, torch.int64: np.int64}

# The sizes that draw() stays under: what the largest listed case of each kind costs.
_LARGEST = {"act": 1 << 24, "bcast": 1 << 24, "stats": 1 << 25, "softmax": 1 << 26, "conv": 1 << 24, "adamw": 25_000_000}


def listed():
    return [
        # a few samples at a time through a classifier: a service answering requests
        {"name": "predict_16", "kind": "predict", "batch": 16, "hidden": 512, "classes": 10, "dtype": "f32"},
        # the repository's own training step: 784-512-512-10, batch 256
        {"name": "train_256", "kind": "train", "batch": 256, "features": 784, "hidden": 512, "classes": 10, "dtype": "f32"},
        # a wider classifier over a data set whose sizes are nobody's choice
        {"name": "train_ragged", "kind": "train", "batch": 1000, "features": 1433, "hidden": 1500, "classes": 999, "dtype": "f32"},
        # an activation on a large tensor, the repository's 2^24 elements
        {"name": "sigmoid_16m", "kind": "act", "fn": "sigmoid", "n": 1 << 24, "dtype": "f32"},
        # broadcasting and transposed operands on the repository's [4096, 4096]
        {"name": "bcast_4096", "kind": "bcast", "rows": 4096, "cols": 4096, "dtype": "f32"},
        # the same on a table of measurements
        {"name": "bcast_ragged", "kind": "bcast", "rows": 3001, "cols": 2047, "dtype": "f32"},
        # statistics of the repository's [8192, 4096]
        {"name": "stats_8192", "kind": "stats", "rows": 8192, "cols": 4096, "dtype": "f32"},
        # statistics of a table of measurements in double precision
        {"name": "stats_ragged", "kind": "stats", "rows": 10007, "cols": 1003, "dtype": "f64"},
        # probabilities over a vocabulary, the longest rows
        {"name": "softmax_vocab", "kind": "softmax", "outer": 2048, "classes": 32003, "inner": 1, "dtype": "f32"},
        # a class per pixel: the softmax axis is not the last one
        {"name": "softmax_pixels", "kind": "softmax", "outer": 16, "classes": 21, "inner": 16384, "dtype": "f32"},
        # a convolution's activations late in an image network: small odd planes, many channels
        {"name": "conv_14", "kind": "conv", "batch": 64, "channels": 512, "height": 14, "width": 14, "dtype": "f32"},
        # 25 million parameters, as a model holds them: a weight and a bias per layer
        {"name": "adamw_25m", "kind": "adamw", "layers": 24, "width": 1020, "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("predict", "train", "act", "bcast", "stats", "softmax", "softmax", "conv", "adamw"))
    dtype = "f64" if rng.random() < 0.25 else "f32"
    case = {"kind": kind, "dtype": dtype}
    most = _LARGEST.get(kind, 0) * 4 // _SIZE[dtype]
    if kind == "predict":
        case.update(batch=_log_int(rng, 1, 512), hidden=_log_int(rng, 64, 4096), classes=_log_int(rng, 10, 1000))
    elif kind == "train":
        case.update(batch=_log_int(rng, 32, 1024), features=_log_int(rng, 64, 1500), hidden=_log_int(rng, 64, 1500),
                    classes=_log_int(rng, 10, 1000))
    elif kind == "act":
        case.update(fn=rng.choice(("relu", "sigmoid", "tanh")), n=_log_int(rng, 1 << 12, most))
    elif kind in ("bcast", "stats"):
        rows = _log_int(rng, 64, 16384)
        case.update(rows=rows, cols=_log_int(rng, 64, min(16384, most // rows)))
    elif kind == "softmax":
        if rng.random() < 0.67:
            classes = _log_int(rng, 10, 50000)
            case.update(outer=_log_int(rng, 16, min(65536, most // classes)), classes=classes, inner=1)
        else:
            classes = _log_int(rng, 2, 512)
            inner = _log_int(rng, 49, 65536 // 4)
            case.update(outer=_log_int(rng, 1, max(1, min(128, most // (4 * classes * inner)))), classes=classes, inner=inner)
    elif kind == "conv":
        side = _log_int(rng, 7, 112)
        channels = _log_int(rng, 3, 512)
        case.update(batch=_log_int(rng, 1, max(1, min(128, most // (channels * side * side)))), channels=channels,
                    height=side, width=side + rng.choice((0, 0, 1)))
    else:
        width = _log_int(rng, 16, 1020)
        case.update(layers=rng.randint(1, max(1, min(40, most // (width * (width + 1))))), width=width)
    return case


# ---- tensors -------------------------------------------------------------------------------------------


class _Memory:
    """torch's memory behind a Matrix: keeps the tensor alive for as long as a view exists"""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


def _matrix(t):
    return Matrix(_Memory(t), 0, tuple(t.shape), zenu.default_stride(tuple(t.shape)), _NUMPY[t.dtype])


class _Make:
    """inputs from one seed, outputs uninitialised; `t` holds the torch tensors by name, `m` the matrices"""

    def __init__(self, case, seed):
        self.dtype = _TORCH[case["dtype"]]
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.t, self.m = {}, {}

    def keep(self, name, tensor):
        self.t[name] = tensor
        self.m[name] = _matrix(tensor)
        return tensor

    def normal(self, name, *shape, scale=1.0, mean=0.0):
        x = torch.empty(shape, dtype=self.dtype, device="cuda").normal_(mean, scale, generator=self.gen)
        return self.keep(name, x)

    def uniform(self, name, *shape):
        return self.keep(name, torch.rand(shape, dtype=self.dtype, device="cuda", generator=self.gen))

    def one_hot(self, name, rows, classes):
        at = torch.randint(classes, (rows, 1), device="cuda", generator=self.gen)
        return self.keep(name, torch.zeros(rows, classes, dtype=self.dtype, device="cuda").scatter_(1, at, 1.0))

    def out(self, name, *shape, dtype=None):
        return self.keep(name, torch.empty(shape, dtype=dtype or self.dtype, device="cuda"))


def _layer_params(k, shapes):
    """Weights and biases as views of one flat parameter store, each tensor at a 256-byte boundary, with
    gradients, first and second moments laid out alike (the distributions of a model in mid-training)."""
    sizes = [int(np.prod(s)) for s in shapes.values()]
    step = 256 // k.dtype.itemsize
    starts, total = [], 0
    for n in sizes:
        starts.append(total)
        total += -(-n // step) * step
    k.normal("p", total, scale=0.02)
    k.normal("g", total, scale=1e-3)
    k.normal("moment1", total, scale=1e-4)
    k.normal("moment2", total, scale=1e-6)
    k.t["moment2"].abs_()
    views = {}
    for what in ("p", "g", "moment1", "moment2"):
        views[what] = {name: _matrix(k.t[what][at:at + n].view(shape))
                       for (name, shape), at, n in zip(shapes.items(), starts, sizes)}
    return views


def _adamw(views):
    weights = [name for name in views["p"] if name.endswith("weight")]
    opt = zenu.AdamW(1e-3, 0.9, 0.999, 1e-8, 0.01, {}, weights)
    opt.m, opt.v, opt.step = views["moment1"], views["moment2"], 9      # resumed from a checkpoint
    return opt


# ---- what a program has in hand before the call -----------------------------------------------------------


def prepare(case, seed):
    k = _Make(case, seed)
    kind = case["kind"]
    state = {"case": dict(case), "code": _CODE[case["dtype"]], "t": k.t, "m": k.m}
    if kind == "predict":
        b, h, c = case["batch"], case["hidden"], case["classes"]
        for i, f in ((1, h), (2, h), (3, c)):
            k.normal(f"z{i}", b, f)
            k.normal(f"b{i}", f, scale=0.1)
        k.out("h1", b, h), k.out("h2", b, h), k.out("logits", b, c), k.out("prob", b, c)
        k.out("label", b, dtype=torch.int64)
    elif kind == "train":
        b, f, h, c = case["batch"], case["features"], case["hidden"], case["classes"]
        # the mini-batch is a run of rows of the data set
        k.uniform("data", b + 1, f)
        k.one_hot("target", b, c)
        # matrix products of the forward and of the backward pass
        k.normal("z1", b, h), k.normal("z2", b, h), k.normal("z3", b, c)
        k.normal("gh1", b, h, scale=1e-3), k.normal("gh2", b, h, scale=1e-3)
        k.normal("gw1", f, h, scale=1e-3), k.normal("gw2", h, h, scale=1e-3), k.normal("gw3", h, c, scale=1e-3)
        views = _layer_params(k, {"l1.weight": (h, f), "l1.bias": (h,), "l2.weight": (h, h), "l2.bias": (h,),
                                  "l3.weight": (c, h), "l3.bias": (c,)})
        for i, (rows, cols) in ((1, (f, h)), (2, (h, h)), (3, (h, c))):
            k.out(f"wt{i}", rows, cols), k.out(f"xt{i}", rows, b)
            k.out(f"wtt{i}", cols, rows)
        for i, w in ((1, h), (2, h)):
            k.out(f"a{i}", b, w), k.out(f"h{i}", b, w), k.out(f"ga{i}", b, w)
        k.out("logits", b, c), k.out("prob", b, c), k.out("glogits", b, c), k.out("loss")
        state.update(opt=_adamw(views), p=views["p"], g=views["g"])
    elif kind == "act":
        k.normal("x", case["n"]), k.normal("gy", case["n"]), k.out("y", case["n"]), k.out("gx", case["n"])
    elif kind == "bcast":
        r, c = case["rows"], case["cols"]
        k.normal("a", r, c), k.normal("b", c, r), k.normal("row", c), k.normal("col", r, 1)
        for name in ("by_row", "by_col", "by_matrix", "by_scalar"):
            k.out(name, r, c)
    elif kind == "stats":
        r, c = case["rows"], case["cols"]
        x = k.normal("x", r, c)
        # about one row in a hundred has its maximum twice
        again = torch.arange(0, r, 100, device="cuda")
        x[again, c - 1] = x[again].max(dim=1).values
        k.out("col_sum", c), k.out("row_sum", r, 1), k.out("row_max", r), k.out("magnitude")
        k.out("row_at", r, dtype=torch.int64)
    elif kind == "softmax":
        shape = (case["outer"], case["classes"]) + ((case["inner"],) if case["inner"] > 1 else ())
        k.normal("x", *shape, scale=3.0), k.normal("gy", *shape, scale=1e-2), k.out("y", *shape), k.out("gx", *shape)
    elif kind == "conv":
        n, c, h, w = case["batch"], case["channels"], case["height"], case["width"]
        k.normal("x", n, c, h, w), k.normal("bias", 1, c, 1, 1), k.normal("gy", n, c, h, w, scale=1e-2)
        for name in ("pre", "y", "gx"):
            k.out(name, n, c, h, w)
        k.out("nhwc", n, h, w, c), k.out("gbias", 1, c, 1, 1)
    else:
        shapes = {}
        for i in range(case["layers"]):
            shapes[f"l{i}.weight"], shapes[f"l{i}.bias"] = (case["width"], case["width"]), (case["width"],)
        views = _layer_params(k, shapes)
        state.update(opt=_adamw(views), p=views["p"], g=views["g"])
    return state


# ---- one pass ------------------------------------------------------------------------------------------------


def _pick(state, *names):
    return {n: state["t"][n] for n in names}


def _call(name, state, *args):
    """a C entry point on the package's stream"""
    args = [C.byref(a.desc()) if isinstance(a, Matrix) else a for a in args]
    _lib.check(getattr(zenu.lib(), name)(state["code"], *args, zenu.get_stream()), name)


def _predict(state, m):
    m["h1"].bias_add_relu(m["z1"], m["b1"], 0.0)
    m["h2"].bias_add_relu(m["z2"], m["b2"], 0.0)
    m["logits"].add_array(m["z3"], m["b3"])
    m["prob"].softmax_assign(m["logits"], 1)
    _call("zenu_hip_max_axis_idx", state, m["label"].as_ptr(), m["prob"], 1)
    return _pick(state, "h1", "h2", "logits", "prob", "label")


def _train(state, m):
    p, g, b = state["p"], state["g"], state["case"]["batch"]
    x = m["data"].slice(slice(1, 1 + b))
    # forward: the transposed weight that the product takes, then bias and ReLU
    m["wt1"].copy_from(p["l1.weight"].transpose())
    m["h1"].bias_add_relu(m["z1"], p["l1.bias"], 0.0, pre=m["a1"])
    m["wt2"].copy_from(p["l2.weight"].transpose())
    m["h2"].bias_add_relu(m["z2"], p["l2.bias"], 0.0, pre=m["a2"])
    m["wt3"].copy_from(p["l3.weight"].transpose())
    m["logits"].add_array(m["z3"], p["l3.bias"])
    _call("zenu_hip_softmax_cross_entropy", state, m["loss"], m["prob"], m["logits"], m["target"])
    # backward: per layer the bias gradient, the transposed input for the weight gradient's product, the
    # weight gradient in the weight's own layout, the transposed weight for the input gradient's product
    _call("zenu_hip_softmax_cross_entropy_backward_bias_grad", state, m["glogits"], g["l3.bias"], m["prob"], m["target"], None)
    for i, inp in ((3, m["h2"]), (2, m["h1"]), (1, x)):
        m[f"xt{i}"].copy_from(inp.transpose())
        g[f"l{i}.weight"].copy_from(m[f"gw{i}"].transpose())
        if i > 1:
            m[f"wtt{i}"].copy_from(m[f"wt{i}"].transpose())
            m[f"ga{i - 1}"].relu_backward_bias_grad(g[f"l{i - 1}.bias"], m[f"gh{i - 1}"], m[f"a{i - 1}"], 0.0)
    state["opt"].update({name: (p[name], g[name]) for name in p})
    return _pick(state, "a1", "h1", "a2", "h2", "logits", "prob", "loss", "glogits", "ga1", "ga2", "wt1", "wt2", "wt3",
                 "xt1", "xt2", "xt3", "wtt2", "wtt3", "p", "g", "moment1", "moment2")


def _act(state, m):
    fn = state["case"]["fn"]
    if fn == "relu":
        m["y"].relu(m["x"], 0.0)
        m["gx"].relu_backward(m["gy"], m["x"], 0.0)
    elif fn == "tanh":
        m["y"].tanh_array(m["x"])
        m["gx"].tanh_backward(m["gy"], m["x"])
    else:
        _lib.check(zenu.lib().zenu_hip_unary(_lib.SIGMOID, state["code"], C.byref(m["y"].desc()), C.byref(m["x"].desc()),
                                             zenu.get_stream()), "sigmoid")
        m["gx"].sigmoid_backward(m["gy"], m["x"])
    return _pick(state, "y", "gx")


def _bcast(state, m):
    m["by_row"].add_array(m["a"], m["row"])
    m["by_col"].mul_array(m["a"], m["col"])
    m["by_matrix"].add_array(m["a"], m["b"].transpose())
    m["by_scalar"].mul_scalar(m["a"], 0.5)
    return _pick(state, "by_row", "by_col", "by_matrix", "by_scalar")


def _stats(state, m):
    zenu.sum_to(m["x"], m["col_sum"])
    zenu.sum_to(m["x"], m["row_sum"])
    _call("zenu_hip_max_axis", state, m["row_max"], m["x"], 1)
    _call("zenu_hip_max_axis_idx", state, m["row_at"].as_ptr(), m["x"], 1)
    _call("zenu_hip_asum", state, m["magnitude"].as_ptr(), m["x"])
    return _pick(state, "col_sum", "row_sum", "row_max", "row_at", "magnitude")


def _softmax(state, m):
    m["y"].softmax_assign(m["x"], 1)
    _call("zenu_hip_softmax_backward", state, m["gx"], m["y"], m["gy"], 1)
    return _pick(state, "y", "gx")


def _conv(state, m):
    zenu.conv2d_bias_add(m["x"], m["bias"], m["pre"])
    m["y"].relu(m["pre"], 0.0)
    m["nhwc"].copy_from(m["y"].transpose_by_index([0, 2, 3, 1]))
    m["gx"].relu_backward(m["gy"], m["pre"], 0.0)
    zenu.conv2d_bias_bkwd(m["gx"], m["gbias"])
    return _pick(state, "pre", "y", "nhwc", "gx", "gbias")


def _optimizer(state, m):
    p, g = state["p"], state["g"]
    state["opt"].update({name: (p[name], g[name]) for name in p})
    return _pick(state, "p", "moment1", "moment2")


_RUN = {"predict": _predict, "train": _train, "act": _act, "bcast": _bcast, "stats": _stats, "softmax": _softmax,
        "conv": _conv, "adamw": _optimizer}


def run(state):
    return _RUN[state["case"]["kind"]](state, state["m"])


# ---- what one pass cannot do without ---------------------------------------------------------------------------


def work(case):
    """Every call reads its operands once and writes its results once."""
    kind, size = case["kind"], _SIZE[case["dtype"]]
    if kind == "predict":
        b, h, c = case["batch"], case["hidden"], case["classes"]
        n = 2 * (2 * b * h + h) + (2 * b * c + c) + 2 * b * c + b * c
        return {"bytes": size * n + 8 * b, "flops": 4 * b * h + 6 * b * c}
    if kind == "train":
        b, f, h, c = case["batch"], case["features"], case["hidden"], case["classes"]
        params = h * f + h + h * h + h + c * h + c
        n = 2 * (3 * b * h + h) + (2 * b * c + c) + 3 * b * c + (3 * b * c + c)       # forward, loss and its backward
        n += 2 * (3 * b * h + h)                                                       # ReLU backward with bias gradients
        n += 2 * (2 * (h * f + h * h + h * c) + h * h + h * c + b * (f + 2 * h))       # transposed copies
        n += 7 * params
        return {"bytes": size * n, "flops": 12 * b * h + 14 * b * c + 14 * params}
    if kind == "act":
        return {"bytes": size * 5 * case["n"], "flops": 2 * case["n"]}
    if kind == "bcast":
        r, c = case["rows"], case["cols"]
        return {"bytes": size * (9 * r * c + r + c), "flops": 4 * r * c}
    if kind == "stats":
        r, c = case["rows"], case["cols"]
        return {"bytes": size * (5 * r * c + c + 2 * r + 1) + 8 * r, "flops": 5 * r * c}
    if kind == "softmax":
        n = case["outer"] * case["classes"] * case["inner"]
        return {"bytes": size * 5 * n, "flops": 8 * n}
    if kind == "conv":
        n = case["batch"] * case["channels"] * case["height"] * case["width"]
        return {"bytes": size * (10 * n + 2 * case["channels"]), "flops": 4 * n}
    n = case["layers"] * case["width"] * (case["width"] + 1)
    return {"bytes": size * 7 * n, "flops": 14 * n}


def tolerance(case):
    """Element by element every result is rounded as the reference rounds it; sums may be taken in another order.
    Against the same pass in f64 (f64: against another order of the sums) the f32 results with sums in them are
    off by up to 2.5e-7 of their norm, f64 ones by 5.5e-16; the softmax gradient, a small difference, by up to
    2e-5 of its root mean square at single elements."""
    if case["kind"] in ("act", "bcast", "adamw"):
        return "exact"
    return {"rel": 1e-6, "max": 8e-5} if case["dtype"] == "f32" else {"rel": 2.2e-15, "max": 2e-13}
