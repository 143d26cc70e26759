"""The work that programs hand to this library, as timed and compared cases.

Every case is a dict of plain values; ``kind`` names the work and the other
fields its sizes and options:

* ``softmax``: a row softmax (or log-softmax) forward and its backward;
* ``reduce``: a matrix summed and averaged whole, and sum / mean / max /
  argmax of its rows and of its columns;
* ``reduce3``: sum, mean, max, argmax and variance over the middle axis of a
  3-D tensor;
* ``affine``: act(X * scale + bias) and its backward, the fused pair;
* ``chain``: the same expression, and more, as separate elementwise calls in
  fp32 (row and column broadcasts among them), bf16 or fp16;
* ``mlp``: one training step of the 3-layer MLP;
* ``linear``: one dense fp32 layer, forward (bias, ReLU) and the three
  gradients of its backward;
* ``matmul16``: a dense layer's three products in bf16 or fp16 (A B, A B^T
  and A^T B as the backward needs them);
* ``xent``: softmax cross-entropy with its gradient, the loss of a
  classifier.

``listed()`` holds the sizes of this repository's own workloads (C1-C5 of
the benchmark) beside small, ragged and many-class ones; ``draw()`` gives
more of the same kinds over their whole ranges.
"""
import math

import torch

from cortexmind_amd import _lib, engine

_ACT = {"relu": engine.ACT_RELU, "sigmoid": engine.ACT_SIGMOID, "tanh": engine.ACT_TANH}
_DTYPE = {"bf16": (torch.bfloat16, _lib.DT_BF16), "f16": (torch.float16, _lib.DT_F16)}
_LR = 0.01


class Buffer:
    """A GPU tensor as the engine's calls take their operands."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.size = tensor.numel()


# ------------------------------------------------------------------ cases


def listed():
    return [
        # the smallest call: attention-sized rows, where launches count (C1)
        {"name": "softmax_512x1024", "kind": "softmax", "rows": 512, "cols": 1024, "log": False, "masked": False},
        # an ordinary batch whose class count is not a multiple of anything
        {"name": "softmax_5000x1003", "kind": "softmax", "rows": 5000, "cols": 1003, "log": False, "masked": False},
        # long rows with a tenth of the entries masked by -inf (C4)
        {"name": "logsoftmax_64x131072", "kind": "softmax", "rows": 64, "cols": 131072, "log": True, "masked": True},
        # statistics of a square activation matrix, whole, by row and by column (C2)
        {"name": "reduce_4096x4096", "kind": "reduce", "rows": 4096, "cols": 4096},
        # statistics over the middle axis, as over the positions of a batch of sequences
        {"name": "reduce3_64x1000x257", "kind": "reduce3", "outer": 64, "dim": 1000, "inner": 257},
        # the largest: a fused scale, shift and activation and its backward (C3)
        {"name": "affine_8192x8192", "kind": "affine", "rows": 8192, "cols": 8192, "act": "tanh"},
        # the same expression and more as separate tensor operators on a ragged matrix
        {"name": "chain_3001x1003", "kind": "chain", "rows": 3001, "cols": 1003, "act": "sigmoid", "dtype": "f32"},
        # a training step at the benchmark's size (C5) ...
        {"name": "mlp_4096", "kind": "mlp", "batch": 4096, "d0": 784, "d1": 1024, "d2": 1024, "d3": 10},
        # ... and at the size of a small batch through a small network
        {"name": "mlp_40", "kind": "mlp", "batch": 40, "d0": 784, "d1": 256, "d2": 256, "d3": 10},
        # a dense layer whose sizes are multiples of nothing
        {"name": "linear_4100x300x4095", "kind": "linear", "m": 4100, "k": 300, "n": 4095},
        # a wide layer in bf16
        {"name": "matmul16_4096x1024x4096", "kind": "matmul16", "m": 4096, "k": 1024, "n": 4096, "dtype": "bf16"},
        # the loss of a thousand-class classifier
        {"name": "xent_4096x1000", "kind": "xent", "batch": 4096, "classes": 1000},
    ]


def _size(rng, low, high):
    """A size spread over the logarithm of [low, high]; about half of the
    larger ones are multiples of 16, as layer widths often are."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if v >= 32 and rng.random() < 0.5:
        v = v // 16 * 16
    return max(low, min(high, v))


def _pair(rng, rows, cols, least, most):
    """(rows, cols) of the two ranges with least <= rows * cols <= most."""
    while True:
        r, c = _size(rng, *rows), _size(rng, *cols)
        if least <= r * c <= most:
            return r, c


def draw(rng):
    kind = rng.choice(["softmax", "reduce", "reduce3", "affine", "chain", "mlp", "linear", "matmul16", "xent"])
    if kind == "softmax":
        r, c = _pair(rng, (1, 65536), (8, 131072), 1 << 15, 64 * 131072)
        return {"kind": kind, "rows": r, "cols": c, "log": rng.random() < 0.5, "masked": rng.random() < 0.3}
    if kind == "reduce":
        r, c = _pair(rng, (4, 262144), (4, 65536), 1 << 15, 4096 * 4096)
        return {"kind": kind, "rows": r, "cols": c}
    if kind == "reduce3":
        while True:
            o, d, i = _size(rng, 1, 512), _size(rng, 8, 4096), _size(rng, 2, 4096)
            if 1 << 15 <= o * d * i <= 4096 * 4096:
                return {"kind": kind, "outer": o, "dim": d, "inner": i}
    if kind == "affine":
        r, c = _pair(rng, (16, 8192), (16, 8192), 1 << 15, 8192 * 8192)
        return {"kind": kind, "rows": r, "cols": c, "act": rng.choice(["relu", "sigmoid", "tanh"])}
    if kind == "chain":
        r, c = _pair(rng, (16, 8192), (16, 8192), 1 << 15, 4096 * 4096)
        return {"kind": kind, "rows": r, "cols": c, "act": rng.choice(["relu", "sigmoid", "tanh"]),
                "dtype": rng.choice(["f32", "f32", "bf16", "f16"])}
    if kind == "mlp":
        return {"kind": kind, "batch": _size(rng, 16, 4096), "d0": _size(rng, 16, 784), "d1": _size(rng, 32, 1024),
                "d2": _size(rng, 32, 1024), "d3": rng.randint(2, 100) if rng.random() < 0.4 else 10}
    if kind == "linear":
        return {"kind": kind, "m": _size(rng, 32, 4100), "k": _size(rng, 32, 1024), "n": _size(rng, 32, 4095)}
    if kind == "matmul16":
        return {"kind": kind, "m": _size(rng, 64, 4096), "k": _size(rng, 64, 1024), "n": _size(rng, 64, 4096),
                "dtype": rng.choice(["bf16", "f16"])}
    r, c = _pair(rng, (64, 16384), (2, 1000), 1 << 10, 4096 * 1000)
    return {"kind": kind, "batch": r, "classes": c}


# ----------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, mean=0.0, std=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=g)


def _uniform(g, shape, low, high):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(low, high, generator=g)


def _labels(g, n, classes):
    return torch.randint(0, classes, (n,), generator=g, device="cuda", dtype=torch.int32)


def _inputs(case, seed):
    """The tensors a program holds before the call."""
    g, kind = _generator(seed), case["kind"]
    if kind == "softmax":
        r, c = case["rows"], case["cols"]
        x = _normal(g, (r, c), 0.0, 8.0 if case["masked"] else 4.0)
        if case["masked"]:
            gone = torch.rand((r, c), generator=g, device="cuda") < 0.1
            gone[:, 0] = False
            x.masked_fill_(gone, -math.inf)
        return {"x": x, "dy": _normal(g, (r, c))}
    if kind == "reduce":
        return {"x": _normal(g, (case["rows"], case["cols"]), 0.5, 1.0)}
    if kind == "reduce3":
        return {"x": _normal(g, (case["outer"], case["dim"], case["inner"]), 0.5, 1.0)}
    if kind == "affine":
        r, c = case["rows"], case["cols"]
        return {"x": _normal(g, (r, c)), "scale": _uniform(g, (c,), 0.5, 1.5), "bias": _normal(g, (c,), 0.0, 0.1),
                "dy": _normal(g, (r, c))}
    if kind == "chain":
        r, c = case["rows"], case["cols"]
        if case["dtype"] == "f32":
            return {"x": _normal(g, (r, c)), "scale": _uniform(g, (c,), 0.5, 1.5), "bias": _normal(g, (c,), 0.0, 0.1),
                    "shift": _normal(g, (r,)), "gain": _normal(g, (r, c), 1.0, 0.1)}
        t = _DTYPE[case["dtype"]][0]
        return {"x": _normal(g, (r, c)).to(t), "y": _normal(g, (r, c)).to(t)}
    if kind == "mlp":
        d = [case["d0"], case["d1"], case["d2"], case["d3"]]
        v = {"x": _uniform(g, (case["batch"], d[0]), 0.0, 1.0), "labels": _labels(g, case["batch"], d[3])}
        for i in range(3):
            v["w%d" % (i + 1)] = _normal(g, (d[i], d[i + 1]), 0.0, math.sqrt(2.0 / d[i]))
            # a network under way: biases away from zero, large beside a step's change
            v["b%d" % (i + 1)] = _normal(g, (d[i + 1],), 0.0, 0.05)
        return v
    if kind in ("linear", "matmul16"):
        m, k, n = case["m"], case["k"], case["n"]
        v = {"x": _normal(g, (m, k)).clamp_(min=0.0), "w": _normal(g, (k, n), 0.0, math.sqrt(2.0 / k)),
             "dz": _normal(g, (m, n))}
        if kind == "linear":
            v["b"] = _normal(g, (n,), 0.0, 0.1)
            return v
        return {name: t.to(_DTYPE[case["dtype"]][0]) for name, t in v.items()}
    return {"logits": _normal(g, (case["batch"], case["classes"]), 0.0, 2.0),
            "labels": _labels(g, case["batch"], case["classes"])}


def prepare(case, seed):
    """Inputs, output buffers and the handle a program keeps."""
    v, kind = _inputs(case, seed), case["kind"]

    def new(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda")

    if kind == "softmax":
        out = {"y": torch.empty_like(v["x"]), "dx": torch.empty_like(v["x"])}
    elif kind == "reduce":
        r, c = case["rows"], case["cols"]
        out = {"sum": new(1), "mean": new(1)}
        for axis, n in (("row", r), ("col", c)):
            out.update({axis + "_sum": new(n), axis + "_mean": new(n), axis + "_max": new(n),
                        axis + "_argmax": new(n, dtype=torch.int32)})
    elif kind == "reduce3":
        o, i = case["outer"], case["inner"]
        out = {"sum": new(o, i), "mean": new(o, i), "max": new(o, i), "argmax": new(o, i, dtype=torch.int32),
               "var": new(o, i)}
    elif kind == "affine":
        c = case["cols"]
        out = {"y": torch.empty_like(v["x"]), "dx": torch.empty_like(v["x"]), "dscale": new(c), "dbias": new(c)}
    elif kind == "chain":
        names = ["scaled", "shifted", "active", "centred", "gained", "halved"] if case["dtype"] == "f32" else \
            ["added", "halved", "active", "squared"]
        out = {name: torch.empty_like(v["x"]) for name in names}
    elif kind == "mlp":
        out = {"loss": new(1)}
    elif kind in ("linear", "matmul16"):
        m, k, n = case["m"], case["k"], case["n"]
        t = v["x"].dtype
        out = {"y": new(m, n, dtype=t), "dx": new(m, k, dtype=t), "dw": new(k, n, dtype=t)}
        if kind == "linear":
            out["db"] = new(n)
    else:
        out = {"loss": new(1), "dlogits": torch.empty_like(v["logits"])}
    state = {"case": case, "out": out}
    state.update({name: Buffer(t) for name, t in v.items()})
    state.update({"_" + name: Buffer(t) for name, t in out.items()})
    if kind == "mlp":
        state["params"] = {name: state[name] for name in ("w1", "b1", "w2", "b2", "w3", "b3")}
        state["net"] = engine.Mlp3(case["batch"], case["d0"], case["d1"], case["d2"], case["d3"])
        out.update({name: b.tensor for name, b in state["params"].items()})
    return state


# -------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    _RUN[case["kind"]](state, case)
    return state["out"]


def _run_softmax(s, case):
    r, c, log = case["rows"], case["cols"], case["log"]
    engine.softmax.forward(s["x"], s["_y"], r, c, log=log)
    engine.softmax.backward(s["_y"], s["dy"], s["_dx"], r, c, log=log)


def _run_reduce(s, case):
    r, c, x, red = case["rows"], case["cols"], s["x"], engine.reduce
    red.sum(x, s["_sum"], r * c)
    red.mean(x, s["_mean"], r * c)
    for axis, sizes in (("_row", (r, c, 1)), ("_col", (1, r, c))):
        red.sum(x, s[axis + "_sum"], *sizes)
        red.mean(x, s[axis + "_mean"], *sizes)
        red.max(x, s[axis + "_max"], *sizes)
        red.argmax(x, s[axis + "_argmax"], *sizes)


def _run_reduce3(s, case):
    sizes, x, red = (case["outer"], case["dim"], case["inner"]), s["x"], engine.reduce
    red.sum(x, s["_sum"], *sizes)
    red.mean(x, s["_mean"], *sizes)
    red.max(x, s["_max"], *sizes)
    red.argmax(x, s["_argmax"], *sizes)
    red.var(x, s["_var"], *sizes)


def _run_affine(s, case):
    r, c, act = case["rows"], case["cols"], _ACT[case["act"]]
    engine.activation.affine_fwd(s["x"], s["scale"], s["bias"], s["_y"], r, c, act)
    engine.activation.affine_bwd(s["x"], s["scale"], s["_y"], s["dy"], s["_dx"], s["_dscale"], s["_dbias"], r, c, act)


def _run_chain(s, case):
    r, c, act = case["rows"], case["cols"], _ACT[case["act"]]
    if case["dtype"] == "f32":
        row, col = engine.Broadcast.row, engine.Broadcast.col
        row.mul(s["x"], s["scale"], s["_scaled"], r, c)
        row.add(s["_scaled"], s["bias"], s["_shifted"], r, c)
        engine.activation.apply(s["_shifted"], s["_active"], r * c, act)
        col.sub(s["_active"], s["shift"], s["_centred"], r, c)
        engine.matrix_t.mul(s["_centred"], s["gain"], s["_gained"], r * c)
        engine.ScalarOp.mul(s["_gained"], 0.5, s["_halved"], r * c)
        return
    n, dt = r * c, _DTYPE[case["dtype"]][1]
    _lib.call("cxm_binary_t", s["x"].ptr, s["y"].ptr, s["_added"].ptr, n, _lib.OP_ADD, dt, None)
    _lib.call("cxm_scalar_t", s["_added"].ptr, 0.5, s["_halved"].ptr, n, _lib.OP_MUL, dt, None)
    _lib.call("cxm_unary_t", s["_halved"].ptr, s["_active"].ptr, n, act, dt, None)
    _lib.call("cxm_wise_t", s["_active"].ptr, s["_squared"].ptr, n, _lib.FN_SQUARE, dt, None)


def _run_mlp(s, case):
    s["net"].step(s["x"], s["labels"], s["params"], _LR, s["_loss"])


def _run_linear(s, case):
    m, k, n = case["m"], case["k"], case["n"]
    engine.gemm(s["x"], s["w"], s["_y"], m, k, n, bias=s["b"], act=engine.ACT_RELU)
    engine.gemm(s["dz"], s["w"], s["_dx"], m, n, k, trans_b=True, gate=s["x"])
    engine.gemm(s["x"], s["dz"], s["_dw"], k, m, n, trans_a=True)
    engine.reduce.sum(s["dz"], s["_db"], 1, m, n)


def _run_matmul16(s, case):
    m, k, n, dt = case["m"], case["k"], case["n"], _DTYPE[case["dtype"]][1]
    engine.matrix_t.matmul_t(s["x"], s["w"], s["_y"], m, k, n, dt)
    _lib.call("cxm_gemm_t", s["dz"].ptr, s["w"].ptr, s["_dx"].ptr, m, n, k, 0, 1, dt, None)
    _lib.call("cxm_gemm_t", s["x"].ptr, s["dz"].ptr, s["_dw"].ptr, k, m, n, 1, 0, dt, None)


def _run_xent(s, case):
    engine.train.softmax_xent(s["logits"], s["labels"], s["_loss"], s["_dlogits"], case["batch"], case["classes"])


_RUN = {"softmax": _run_softmax, "reduce": _run_reduce, "reduce3": _run_reduce3, "affine": _run_affine,
        "chain": _run_chain, "mlp": _run_mlp, "linear": _run_linear, "matmul16": _run_matmul16, "xent": _run_xent}


# ------------------------------------------------------- work, tolerances


def work(case):
    """Compulsory traffic of a pass (per call: each input read once, each
    output written once) and the operations of its products."""
    kind = case["kind"]
    if kind == "softmax":
        return {"bytes": 20 * case["rows"] * case["cols"], "flops": 0}
    if kind == "reduce":
        r, c = case["rows"], case["cols"]
        return {"bytes": 4 * (10 * r * c + 4 * (r + c) + 2), "flops": 0}
    if kind == "reduce3":
        o, d, i = case["outer"], case["dim"], case["inner"]
        return {"bytes": 4 * 5 * (o * d * i + o * i), "flops": 0}
    if kind == "affine":
        r, c = case["rows"], case["cols"]
        return {"bytes": 4 * (6 * r * c + 5 * c), "flops": 0}
    if kind == "chain":
        r, c = case["rows"], case["cols"]
        if case["dtype"] == "f32":
            return {"bytes": 4 * (13 * r * c + 2 * c + r), "flops": 0}
        return {"bytes": 2 * 9 * r * c, "flops": 0}
    if kind == "mlp":
        b, d0, d1, d2, d3 = (case[k] for k in ("batch", "d0", "d1", "d2", "d3"))
        weights = d0 * d1 + d1 * d2 + d2 * d3
        return {"bytes": 4 * (b * (d0 + 1) + 2 * (weights + d1 + d2 + d3)),
                "flops": 2 * b * (2 * weights + d1 * d2 + d2 * d3)}
    if kind in ("linear", "matmul16"):
        m, k, n = case["m"], case["k"], case["n"]
        size = 4 if kind == "linear" else 2
        return {"bytes": size * 3 * (m * k + k * n + m * n), "flops": 6 * m * k * n}
    return {"bytes": 4 * (2 * case["batch"] * case["classes"] + case["batch"]), "flops": 0}


def tolerance(case):
    """Largest error of another correct implementation: about four times what
    this one shows against 64 bits over the listed cases and 90 drawn ones
    (in brackets; 16-bit kinds: the rounding of the type)."""
    kind = case["kind"]
    if kind == "chain" and case["dtype"] != "f32":  # [bf16 4e-3, f16 5.2e-4, over the two roundings of the square]
        return {"rel": 1.6e-2 if case["dtype"] == "bf16" else 2e-3}
    if kind == "matmul16":  # [bf16 1.7e-3, f16 2.1e-4]
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 9e-4}
    if kind == "softmax":  # [4.8e-7; single values of dx, where dy and its row's sum cancel, 6.1e-5]
        return {"rel": 2e-6, "max": 2.5e-4}
    if kind in ("reduce", "reduce3"):  # [1.5e-7]
        return {"rel": 6e-7}
    if kind == "affine":  # [2.5e-7]
        return {"rel": 1e-6}
    if kind == "chain":  # [4.2e-8: three or four roundings]
        return {"rel": 1.7e-7}
    if kind == "mlp":  # [1e-6; single values: a unit within rounding of the ReLU's kink]
        return {"rel": 4e-6, "max": 1.5e-4}
    if kind == "linear":  # [8.1e-7: k-term sums in fp32]
        return {"rel": 3e-6}
    return {"rel": 4e-7}  # xent [8.5e-8]


# ------------------------------------------------------------ in 64 bits


def _d(t):
    return t.double()


def exact(case, seed):
    v, kind = _inputs(case, seed), case["kind"]
    if kind == "softmax":
        x, dy = _d(v["x"]), _d(v["dy"])
        if case["log"]:
            y = torch.log_softmax(x, 1)
            return {"y": y, "dx": dy - y.exp() * dy.sum(1, keepdim=True)}
        y = torch.softmax(x, 1)
        return {"y": y, "dx": y * (dy - (dy * y).sum(1, keepdim=True))}
    if kind == "reduce":
        x = _d(v["x"])
        out = {"sum": x.sum().reshape(1), "mean": x.mean().reshape(1)}
        for axis, d in (("row", 1), ("col", 0)):
            out.update({axis + "_sum": x.sum(d), axis + "_mean": x.mean(d), axis + "_max": x.amax(d),
                        axis + "_argmax": None})
        return out
    if kind == "reduce3":
        x = _d(v["x"])
        return {"sum": x.sum(1), "mean": x.mean(1), "max": x.amax(1), "argmax": None,
                "var": x.var(1, unbiased=False)}
    if kind == "affine":
        x, scale, dy = _d(v["x"]), _d(v["scale"]), _d(v["dy"])
        y, slope = _act(case["act"], x * scale + _d(v["bias"]))
        dz = dy * slope
        return {"y": y, "dx": dz * scale, "dscale": (dz * x).sum(0), "dbias": dz.sum(0)}
    if kind == "chain":
        if case["dtype"] == "f32":
            out = {"scaled": _d(v["x"]) * _d(v["scale"])}
            out["shifted"] = out["scaled"] + _d(v["bias"])
            out["active"] = _act(case["act"], out["shifted"])[0]
            out["centred"] = out["active"] - _d(v["shift"])[:, None]
            out["gained"] = out["centred"] * _d(v["gain"])
            out["halved"] = out["gained"] * 0.5
            return out
        out = {"added": _d(v["x"]) + _d(v["y"])}
        out["halved"] = out["added"] * 0.5
        out["active"] = _act(case["act"], out["halved"])[0]
        out["squared"] = out["active"] * out["active"]
        return out
    if kind == "mlp":
        return _exact_mlp(case, v)
    if kind in ("linear", "matmul16"):
        x, w, dz = _d(v["x"]), _d(v["w"]), _d(v["dz"])
        out = {"y": x @ w, "dx": dz @ w.t().contiguous(), "dw": x.t().contiguous() @ dz}
        if kind == "linear":
            out["y"] = (out["y"] + _d(v["b"])).clamp_(min=0.0)
            out["dx"] = out["dx"] * (x > 0)
            out["db"] = dz.sum(0)
        return out
    z, lab = _d(v["logits"]), v["labels"].long()
    loss, dz = _xent(z, lab)
    return {"loss": loss, "dlogits": dz}


def _act(name, t):
    """(act(t), its slope)."""
    if name == "relu":
        y = t.clamp(min=0.0)
        return y, (y > 0).double()
    if name == "sigmoid":
        y = torch.sigmoid(t)
        return y, y * (1.0 - y)
    y = torch.tanh(t)
    return y, 1.0 - y * y


def _xent(z, lab):
    rows = torch.arange(z.shape[0], device=z.device)
    logp = torch.log_softmax(z, 1)
    dz = logp.exp()
    dz[rows, lab] -= 1.0
    return -logp[rows, lab].mean().reshape(1), dz / z.shape[0]


def _exact_mlp(case, v):
    x, lab = _d(v["x"]), v["labels"].long()
    w = [_d(v["w%d" % i]) for i in (1, 2, 3)]
    b = [_d(v["b%d" % i]) for i in (1, 2, 3)]
    h1 = (x @ w[0] + b[0]).clamp_(min=0.0)
    h2 = (h1 @ w[1] + b[1]).clamp_(min=0.0)
    loss, dz = _xent(h2 @ w[2] + b[2], lab)
    dh2 = (dz @ w[2].t().contiguous()) * (h2 > 0)
    dh1 = (dh2 @ w[1].t().contiguous()) * (h1 > 0)
    out = {"loss": loss}
    for i, (a, g) in enumerate(((x, dh1), (h1, dh2), (h2, dz))):
        out["w%d" % (i + 1)] = w[i] - _LR * (a.t().contiguous() @ g)
        out["b%d" % (i + 1)] = b[i] - _LR * g.sum(0)
    return out
