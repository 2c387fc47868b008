"""The workloads this library is timed on: single layers and one training step,
called through the public entry points as a training program calls them.

A program that trains with this library holds fp32 tensors on the GPU and
either queues the ``*_async`` calls of the C ABI on its stream (through
``ml_framework_amd.capi``) or calls the ``seera_cuda`` module, whose functions
return when their result is ready. Every state here keeps what such a program
keeps: the inputs, the output buffers and the stream handle.

Kinds of case (``case["kind"]``):
  dense   a Dense layer: forward with bias and ReLU, backward with the input's
          ReLU mask and the bias gradient
  mlp     a whole step of a three-layer classifier through ``seera_cuda``
  gemm    a matrix product, forward alone or with both gradients
  conv    a Conv2D layer, plain or with bias and ReLU, forward and backward
  convt   a ConvTranspose2D layer, forward and backward
  block   a small image classifier's block: MaxPool, then Conv2D + bias + ReLU,
          forward and backward

Operands of the products are rounded to fp16 (nearest even) and accumulated in
fp32: that rounding is part of what the entry points promise, so ``exact``
rounds the same operands and does the rest in 64 bits.
"""
from __future__ import annotations

import math

import torch

import ml_framework_amd
from ml_framework_amd import capi

RELU = capi.SEERA_ACT_RELU


def listed():
    return [
        # The first layer of an MNIST classifier at batch 64: 784 pixels to 128
        # units. The smallest calls a program makes: launches and latency.
        {"name": "dense_64x784x128", "kind": "dense", "rows": 64, "inputs": 784, "outputs": 128},
        # A training step of the 784-512-256-10 classifier at batch 256, call
        # by call as the Python front end runs it (each call synchronous).
        {"name": "mlp_step", "kind": "mlp", "batch": 256, "inputs": 784, "hidden1": 512, "hidden2": 256, "classes": 10},
        # The square product that large dense layers are judged by.
        {"name": "gemm_4096", "kind": "gemm", "batch": 1, "m": 4096, "n": 4096, "k": 4096, "backward": False},
        # Sides that are no multiple of anything, with both gradients.
        {"name": "gemm_odd", "kind": "gemm", "batch": 1, "m": 3001, "n": 2047, "k": 1501, "backward": True},
        # A sequence batch through one shared weight, with both gradients.
        {"name": "gemm_16x512", "kind": "gemm", "batch": 16, "m": 512, "n": 512, "k": 512, "backward": True},
        # The second block of a small image classifier on 28 x 28 images.
        {"name": "block_28", "kind": "block", "batch": 64, "c": 32, "f": 64, "h": 28, "w": 28},
        # The 3x3 layers of a residual network's four stages; the first is the
        # largest call of such a network at batch 128, the last two have many
        # channels on rows that are no multiple of four.
        {"name": "conv3x3_56", "kind": "conv", "batch": 128, "c": 64, "h": 56, "w": 56, "f": 64, "k": 3, "stride": 1, "pad": 1, "bias": False},
        {"name": "conv3x3_14", "kind": "conv", "batch": 64, "c": 256, "h": 14, "w": 14, "f": 256, "k": 3, "stride": 1, "pad": 1, "bias": True},
        # The layer that halves the image between two stages.
        {"name": "conv3x3_s2", "kind": "conv", "batch": 64, "c": 128, "h": 28, "w": 28, "f": 256, "k": 3, "stride": 2, "pad": 1, "bias": False},
        # The projection of a bottleneck block.
        {"name": "conv1x1_56", "kind": "conv", "batch": 64, "c": 256, "h": 56, "w": 56, "f": 64, "k": 1, "stride": 1, "pad": 0, "bias": False},
        # The stem: 7x7 with stride 2 on colour images.
        {"name": "conv7x7_stem", "kind": "conv", "batch": 32, "c": 3, "h": 224, "w": 224, "f": 64, "k": 7, "stride": 2, "pad": 3, "bias": False},
        # The up-sampling layer of a decoder.
        {"name": "convt4x4_28", "kind": "convt", "batch": 32, "c": 128, "h": 28, "w": 28, "f": 64, "k": 4, "stride": 2, "pad": 1},
    ]


# A drawn case does no more than the largest listed one (gemm_4096's 137 GFLOP,
# conv3x3_56's 89 GFLOP and 617 MB).
MOST_GEMM_FLOPS = 137e9
MOST_CONV_FLOPS = 88e9
MOST_CONV_BYTES = 600e6


def _log(rng, low, high, step=1):
    """A size spread evenly over the logarithm of [low, high]."""
    v = math.exp(rng.uniform(math.log(low), math.log(high + 1)))
    return max(low, min(high, int(v) // step * step))


def _draw_once(rng):
    kind = rng.choice(["dense", "mlp", "gemm", "gemm", "conv", "conv", "conv", "conv", "convt", "block"])
    if kind == "dense":
        return {"kind": kind, "rows": _log(rng, 16, 1024), "inputs": _log(rng, 32, 2048), "outputs": _log(rng, 10, 1024)}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 16, 512), "inputs": _log(rng, 64, 1024), "hidden1": _log(rng, 64, 1024),
                "hidden2": _log(rng, 32, 512), "classes": rng.randint(2, 100)}
    if kind == "gemm":
        batch = rng.choice([1, 1, 1, rng.randint(2, 16)])
        step = rng.choice([1, 1, 4, 64])
        top = 4096 if batch == 1 else 1024
        m, n, k = (_log(rng, 64, top, step) for _ in range(3))
        return {"kind": kind, "batch": batch, "m": m, "n": n, "k": k, "backward": rng.random() < 0.7}
    if kind == "block":
        side = rng.choice([28, 32, rng.randint(16, 48) // 2 * 2])
        return {"kind": kind, "batch": _log(rng, 8, 256), "c": rng.choice([8, 16, 32]), "f": rng.choice([16, 32, 64]), "h": side, "w": side}
    if kind == "convt":
        side = _log(rng, 4, 56)
        return {"kind": kind, "batch": _log(rng, 4, 64), "c": 16 * _log(rng, 1, 16), "h": side, "w": side, "f": 16 * _log(rng, 1, 8),
                "k": 4, "stride": 2, "pad": 1}
    form = rng.choice(["3x3", "3x3", "3x3", "s2", "s2", "1x1", "1x1", "stem", "first"])
    if form == "first":  # a small classifier's first layer
        side = rng.choice([28, 32, 64, _log(rng, 16, 112)])
        return {"kind": kind, "batch": _log(rng, 8, 128), "c": rng.choice([1, 3]), "h": side, "w": side, "f": rng.choice([8, 16, 32, 64]),
                "k": 3, "stride": 1, "pad": 1, "bias": True}
    if form == "stem":
        side = rng.choice([96, 112, 128, 160, 192, 224])
        return {"kind": kind, "batch": _log(rng, 4, 32), "c": rng.choice([1, 3]), "h": side, "w": side, "f": rng.choice([32, 64]),
                "k": 7, "stride": 2, "pad": 3, "bias": rng.random() < 0.5}
    # stages of a residual network, their channels and the sizes around them
    side = rng.choice([7, 14, 28, 56, _log(rng, 7, 112), _log(rng, 7, 112)])
    c = rng.choice([32, 64, 128, 256, 512, 8 * _log(rng, 2, 64)])
    f = c if form == "3x3" and rng.random() < 0.6 else rng.choice([32, 64, 128, 256, 512, 8 * _log(rng, 2, 64)])
    return {"kind": kind, "batch": _log(rng, 8, 128), "c": c, "h": side, "w": side, "f": f, "k": 1 if form == "1x1" else 3,
            "stride": 2 if form == "s2" else 1, "pad": 0 if form == "1x1" else 1, "bias": rng.random() < 0.5}


def draw(rng):
    """One more case of the same kinds and ranges."""
    while True:
        case = _draw_once(rng)
        w = work(case)
        if case["kind"] in ("conv", "convt"):
            if w["flops"] <= MOST_CONV_FLOPS and w["bytes"] <= MOST_CONV_BYTES:
                return case
        elif w["flops"] <= MOST_GEMM_FLOPS:
            return case


# ---- shapes and work ----


def _out_side(case):
    """Output height and width of a conv / convt case."""
    k, s, p = case["k"], case["stride"], case["pad"]
    if case["kind"] == "convt":
        return (case["h"] - 1) * s - 2 * p + k, (case["w"] - 1) * s - 2 * p + k
    return (case["h"] + 2 * p - k) // s + 1, (case["w"] + 2 * p - k) // s + 1


def _layers(case):
    return [case["inputs"], case["hidden1"], case["hidden2"], case["classes"]]


def work(case):
    """fp32 bytes with each input of the pass read once and each output written
    once, and 2 FLOP for each multiply-add of the products."""
    kind = case["kind"]
    if kind == "dense":
        m, k, n = case["rows"], case["inputs"], case["outputs"]
        # in: x, its mask, w, b, dY; out: y, its mask, dX, dW, db
        return {"bytes": 4 * (3 * m * k + 2 * k * n + 2 * n + 3 * m * n), "flops": 6 * m * n * k}
    if kind == "mlp":
        sizes, b = _layers(case), case["batch"]
        params = sum(i * o + o for i, o in zip(sizes, sizes[1:]))
        products = sum(i * o for i, o in zip(sizes, sizes[1:]))
        # in: x, labels, parameters; out: logits and the gradients
        return {"bytes": 4 * (b * sizes[0] + 2 * b * sizes[-1] + 2 * params),
                "flops": 6 * b * products - 2 * b * sizes[0] * sizes[1]}
    if kind == "gemm":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        a, w, c = b * m * k, k * n, b * m * n
        if not case["backward"]:
            return {"bytes": 4 * (a + w + c), "flops": 2 * b * m * n * k}
        return {"bytes": 4 * (2 * a + 2 * w + 2 * c), "flops": 6 * b * m * n * k}
    if kind == "block":
        b, c, f, h, w = (case[x] for x in ("batch", "c", "f", "h", "w"))
        x, q, y = b * c * h * w, b * c * (h // 2) * (w // 2), b * f * (h // 2) * (w // 2)
        # in: x, w, bias, dY; out: the pooled x, the pool's mask, y, its ReLU mask, d(pooled x), dX, dW, db
        return {"bytes": 4 * (3 * x + 2 * q + 3 * y + 2 * 9 * f * c + 2 * f), "flops": 3 * 2 * 9 * f * c * b * (h // 2) * (w // 2)}
    b, c, f, k = (case[x] for x in ("batch", "c", "f", "k"))
    ho, wo = _out_side(case)
    x, y, w = b * c * case["h"] * case["w"], b * f * ho * wo, f * c * k * k
    taps_over = x * f if kind == "convt" else y * c
    more = (y + 2 * f) if case.get("bias") else 0  # the ReLU mask, the bias and its gradient
    return {"bytes": 4 * (2 * x + 2 * y + 2 * w + more), "flops": 3 * 2 * taps_over * k * k}


# About four times the largest difference to ``exact`` seen over the listed and
# 120 drawn cases of each kind (in brackets): fp32 sums of up to 400 thousand
# products in one order or another. ReLU masks are whole numbers; a few may
# differ where a sum lies within rounding of zero (3e-7 of them seen).
TOLERANCE = {
    "dense": {"rel": 2e-6, "differ": 1e-4},  # 1.3e-7, and longer sums in one chain
    # three layers, each rounding its fp32 input to fp16: a sum that lands on
    # the other side of a rounding boundary travels on as one fp16 ulp (7.4e-5)
    "mlp": {"rel": 3e-4},
    "gemm": {"rel": 2e-6},  # 4.1e-7
    "conv": {"rel": 2e-6, "differ": 1e-4},  # 4.3e-7
    "convt": {"rel": 2e-6},  # 3.1e-7
    "block": {"rel": 2e-6, "differ": 1e-4},  # 1.8e-7, and longer sums in one chain
}


def tolerance(case):
    return dict(TOLERANCE[case["kind"]])


# ---- inputs ----


class _Inputs:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.device = torch.device("cuda")
        self.gen = torch.Generator(device=self.device).manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device=self.device).mul_(scale)

    def uniform(self, *shape, low=-1.0, high=1.0):
        return torch.rand(*shape, generator=self.gen, device=self.device).mul_(high - low).add_(low)

    def kaiming(self, *shape, fan_in):
        limit = math.sqrt(6.0 / fan_in)
        return self.uniform(*shape, low=-limit, high=limit)

    def integers(self, high, *shape):
        return torch.randint(high, shape, generator=self.gen, device=self.device)


def _inputs(case, seed):
    """The tensors a program has in hand before the call."""
    kind, r = case["kind"], _Inputs(seed)
    if kind == "dense":
        m, k, n = case["rows"], case["inputs"], case["outputs"]
        x = r.normal(m, k).relu_()  # what the ReLU before this layer gave
        return {"x": x, "xmask": (x > 0).float(), "w": r.kaiming(k, n, fan_in=k), "b": r.normal(n, scale=0.1), "dy": r.normal(m, n)}
    if kind == "mlp":
        sizes, b = _layers(case), case["batch"]
        t = {"x": r.uniform(b, sizes[0], low=0.0), "onehot": torch.zeros(b, sizes[-1], device=r.device)}
        t["onehot"].scatter_(1, r.integers(sizes[-1], b, 1), 1.0)
        for i, (a, o) in enumerate(zip(sizes, sizes[1:])):
            t["w%d" % i], t["b%d" % i] = r.kaiming(a, o, fan_in=a), r.normal(o, scale=0.1)
        return t
    if kind == "gemm":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        t = {"a": r.uniform(b, m, k), "b": r.uniform(k, n)}
        if case["backward"]:
            t["dc"] = r.uniform(b, m, n)
        return t
    if kind == "block":
        b, c, f, h, w = (case[x] for x in ("batch", "c", "f", "h", "w"))
        x = r.normal(b, c, h, w).relu_()  # what the layer before gave
        return {"x": x, "w": r.kaiming(f, c, 3, 3, fan_in=9 * c), "b": r.normal(f, scale=0.1), "dy": r.normal(b, f, h // 2, w // 2)}
    b, c, f, k = (case[x] for x in ("batch", "c", "f", "k"))
    ho, wo = _out_side(case)
    x = r.normal(b, c, case["h"], case["w"])
    if kind == "convt":
        return {"x": x, "w": r.kaiming(c, f, k, k, fan_in=c * k * k), "dy": r.normal(b, f, ho, wo)}
    return {"x": x, "w": r.kaiming(f, c, k, k, fan_in=c * k * k), "b": r.normal(f, scale=0.1), "dy": r.normal(b, f, ho, wo)}


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    like = torch.empty_like
    if kind == "dense":
        t.update(y=like(t["dy"]), ymask=like(t["dy"]), dx=like(t["x"]), dw=like(t["w"]), db=like(t["b"]))
    elif kind == "mlp":
        sizes, b = _layers(case), case["batch"]
        for i, (a, o) in enumerate(zip(sizes, sizes[1:])):
            for name in ("p%d", "z%d", "h%d", "g%d", "dz%d"):  # product, + bias, ReLU, its gradient, dLoss/dz
                t[name % i] = torch.empty(b, o, device="cuda")
            t["dh%d" % i] = torch.empty(b, a, device="cuda")
            t["dw%d" % i], t["db%d" % i] = like(t["w%d" % i]), like(t["b%d" % i])
        t["prob"] = like(t["onehot"])
        t["module"] = ml_framework_amd.seera_cuda()
    elif kind == "gemm":
        t["c"] = torch.empty(case["batch"], case["m"], case["n"], device="cuda")
        if case["backward"]:
            t.update(da=like(t["a"]), db=like(t["b"]))
    elif kind == "block":
        q = torch.empty(case["batch"], case["c"], case["h"] // 2, case["w"] // 2, device="cuda")
        t.update(q=q, qmask=torch.empty(t["x"].shape, dtype=torch.int32, device="cuda"), y=like(t["dy"]), ymask=like(t["dy"]), dq=like(q),
                 dx=like(t["x"]), dw=like(t["w"]), db=like(t["b"]))
    else:
        t.update(y=like(t["dy"]), dx=like(t["x"]), dw=like(t["w"]))
        if case.get("bias"):
            t.update(ymask=like(t["dy"]), db=like(t["b"]))
    # the pointers and the stream, as a program that drives a C ABI holds them
    ptr = {name: v.data_ptr() for name, v in t.items() if isinstance(v, torch.Tensor)}
    return {"case": case, "t": t, "p": ptr, "stream": torch.cuda.current_stream().cuda_stream}


# ---- the calls ----


def _bits(mask):
    """A ReLU mask's 0.0 / 1.0 as whole numbers (a view of the same memory)."""
    return mask.view(torch.int32)


def _run_dense(case, t, p, stream):
    m, k, n = case["rows"], case["inputs"], case["outputs"]
    capi.call("seera_hip_matmul_bias_act_async", p["x"], p["w"], p["b"], p["y"], p["ymask"], m, n, k, 1, RELU, stream)
    capi.call("seera_hip_matmul_bwd_relu_bias_async", p["x"], p["w"], p["dy"], p["xmask"], p["dx"], p["dw"], p["db"], m, n, k, 1, stream)
    return {"y": t["y"], "ymask": _bits(t["ymask"]), "dx": t["dx"], "dw": t["dw"], "db": t["db"]}


def _run_mlp(case, t, p, stream):
    sc, b, sizes = t["module"], case["batch"], _layers(case)
    h = p["x"]
    for i, (a, o) in enumerate(zip(sizes, sizes[1:])):
        sc.cuda_matmul(h, p["w%d" % i], p["p%d" % i], b, o, a, 1)
        sc.broadcast_add_4d(p["p%d" % i], p["b%d" % i], p["z%d" % i], 1, 1, b, o, 1, 1, 1, o)
        if i < 2:
            sc.cuda_relu_fwd(p["z%d" % i], p["h%d" % i], p["g%d" % i], b * o)
        h = p["h%d" % i]
    sc.cuda_softmax_fwd(p["z2"], p["prob"], b, sizes[-1])
    sc.cuda_elemsub(p["prob"], p["onehot"], p["dz2"], b * sizes[-1])
    sc.cuda_scaler_multiply_f(p["dz2"], 1.0 / b, b * sizes[-1])
    for i in (2, 1, 0):
        a, o = sizes[i], sizes[i + 1]
        sc.cuda_matmul_bwd(p["h%d" % (i - 1)] if i else p["x"], p["w%d" % i], p["dz%d" % i], p["dh%d" % i], p["dw%d" % i], b, o, a, 1)
        sc.cuda_bias_grad(p["dz%d" % i], p["db%d" % i], b, o)
        if i:
            sc.cuda_elemmult(p["dh%d" % i], p["g%d" % (i - 1)], p["dz%d" % (i - 1)], b * a)
    return {"logits": t["z2"], "prob": t["prob"], "dx": t["dh0"], **{n + str(i): t[n + str(i)] for i in range(3) for n in ("dw", "db")}}


def _run_gemm(case, t, p, stream):
    b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
    capi.call("seera_hip_matmul_async", p["a"], p["b"], p["c"], m, n, k, b, stream)
    if not case["backward"]:
        return {"c": t["c"]}
    capi.call("seera_hip_matmul_bwd_async", p["a"], p["b"], p["dc"], p["da"], p["db"], m, n, k, b, stream)
    return {"c": t["c"], "da": t["da"], "db": t["db"]}


def _run_block(case, t, p, stream):
    b, c, f, h, w = (case[x] for x in ("batch", "c", "f", "h", "w"))
    i, j = h // 2, w // 2
    capi.call("seera_hip_maxpool_fwd_async", p["x"], p["q"], p["qmask"], b, c, h, w, 2, 2, 0, 0, 2, 2, stream)
    capi.call("seera_hip_conv2d_fwd_bias_act_async", p["q"], p["w"], p["b"], p["y"], p["ymask"], b, c, i, j, f, 3, 3, 1, 1, 1, 1, RELU, stream)
    capi.call("seera_hip_conv2d_bwd_bias_async", p["w"], p["q"], p["dy"], p["dq"], p["dw"], p["db"], b, c, i, j, f, 3, 3, 1, 1, 1, 1, stream)
    capi.call("seera_hip_maxpool_bwd_async", p["dq"], p["qmask"], p["dx"], b, c, h, w, 2, 2, 0, 0, 2, 2, stream)
    return {"q": t["q"], "qmask": t["qmask"], "y": t["y"], "ymask": _bits(t["ymask"]), "dq": t["dq"], "dx": t["dx"], "dw": t["dw"], "db": t["db"]}


def _run_conv(case, t, p, stream):
    b, c, h, w, f, k, s, q = (case[x] for x in ("batch", "c", "h", "w", "f", "k", "stride", "pad"))
    # the forward takes pad before stride, the backward stride before pad
    if case["bias"]:
        capi.call("seera_hip_conv2d_fwd_bias_act_async", p["x"], p["w"], p["b"], p["y"], p["ymask"], b, c, h, w, f, k, k, q, q, s, s, RELU, stream)
        capi.call("seera_hip_conv2d_bwd_bias_async", p["w"], p["x"], p["dy"], p["dx"], p["dw"], p["db"], b, c, h, w, f, k, k, s, s, q, q, stream)
        return {"y": t["y"], "ymask": _bits(t["ymask"]), "dx": t["dx"], "dw": t["dw"], "db": t["db"]}
    capi.call("seera_hip_conv2d_fwd_async", p["x"], p["w"], p["y"], b, c, h, w, f, k, k, q, q, s, s, stream)
    capi.call("seera_hip_conv2d_bwd_async", p["w"], p["x"], p["dy"], p["dx"], p["dw"], b, c, h, w, f, k, k, s, s, q, q, stream)
    return {"y": t["y"], "dx": t["dx"], "dw": t["dw"]}


def _run_convt(case, t, p, stream):
    b, c, h, w, f, k, s, q = (case[x] for x in ("batch", "c", "h", "w", "f", "k", "stride", "pad"))
    capi.call("seera_hip_conv2DTranpose_fwd_async", p["x"], p["w"], p["y"], b, c, h, w, f, k, k, s, s, q, q, stream)
    capi.call("seera_hip_conv2DTranspose_bwd_async", p["w"], p["x"], p["dy"], p["dx"], p["dw"], b, c, h, w, f, k, k, s, s, q, q, stream)
    return {"y": t["y"], "dx": t["dx"], "dw": t["dw"]}


_RUN = {"dense": _run_dense, "mlp": _run_mlp, "gemm": _run_gemm, "block": _run_block, "conv": _run_conv, "convt": _run_convt}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](case, state["t"], state["p"], state["stream"])


# ---- the same in 64 bits ----


def _h(x):
    """An operand of a product: rounded to fp16, then 64 bits."""
    return x.half().double()


def _taps(x, k, stride, pad, ho, wo):
    """For each kernel tap (r, s): the padded input's values under it, [B, C, Ho * Wo]."""
    xp = torch.nn.functional.pad(x, (pad, pad, pad, pad))
    for r in range(k):
        for s in range(k):
            v = xp[:, :, r:r + stride * (ho - 1) + 1:stride, s:s + stride * (wo - 1) + 1:stride]
            yield r, s, v.reshape(x.shape[0], x.shape[1], ho * wo)


def _conv_fwd(x, w, stride, pad):
    b, _, h, wd = x.shape
    f, _, k, _ = w.shape
    ho, wo = (h + 2 * pad - k) // stride + 1, (wd + 2 * pad - k) // stride + 1
    y = torch.zeros(b, f, ho * wo, dtype=torch.float64, device=x.device)
    for r, s, v in _taps(x, k, stride, pad, ho, wo):
        y += torch.matmul(w[:, :, r, s].contiguous(), v)
    return y.view(b, f, ho, wo)


def _conv_dx(dy, w, stride, pad, h, wd):
    b, f, ho, wo = dy.shape
    _, c, k, _ = w.shape
    dxp = torch.zeros(b, c, h + 2 * pad, wd + 2 * pad, dtype=torch.float64, device=dy.device)
    flat = dy.reshape(b, f, ho * wo)
    for r in range(k):
        for s in range(k):
            dxp[:, :, r:r + stride * (ho - 1) + 1:stride, s:s + stride * (wo - 1) + 1:stride] += torch.matmul(
                w[:, :, r, s].t().contiguous(), flat).view(b, c, ho, wo)
    return dxp[:, :, pad:pad + h, pad:pad + wd].contiguous()


def _conv_dw(dy, x, k, stride, pad):
    b, f, ho, wo = dy.shape
    c = x.shape[1]
    dw = torch.zeros(f, c, k, k, dtype=torch.float64, device=dy.device)
    left = dy.permute(1, 0, 2, 3).reshape(f, b * ho * wo)
    for r, s, v in _taps(x, k, stride, pad, ho, wo):
        dw[:, :, r, s] = left @ v.permute(0, 2, 1).reshape(b * ho * wo, c).contiguous()
    return dw


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "dense":
        pre = _h(t["x"]) @ _h(t["w"]) + t["b"].double()
        return {"y": pre.relu(), "ymask": _bits((pre > 0).float()), "dx": (_h(t["dy"]) @ _h(t["w"]).t()) * t["xmask"].double(),
                "dw": _h(t["x"]).t() @ _h(t["dy"]), "db": t["dy"].double().sum(0)}
    if kind == "mlp":
        h, acts, masks = t["x"].double(), [t["x"].double()], []
        for i in range(3):
            z = _h(h) @ _h(t["w%d" % i]) + t["b%d" % i].double()
            h = z.relu()
            acts.append(h)
            masks.append((z > 0).double())
        out = {"logits": z, "prob": torch.softmax(z, 1)}
        dz = (out["prob"] - t["onehot"].double()) / case["batch"]
        for i in (2, 1, 0):
            out["dw%d" % i], out["db%d" % i] = _h(acts[i]).t() @ _h(dz), dz.sum(0)
            dh = _h(dz) @ _h(t["w%d" % i]).t()
            dz = dh * masks[i - 1] if i else None
        out["dx"] = dh
        return out
    if kind == "gemm":
        a, b = _h(t["a"]), _h(t["b"])
        c = torch.stack([one @ b for one in a])
        if not case["backward"]:
            return {"c": c}
        dc = _h(t["dc"])
        da = torch.stack([one @ b.t() for one in dc])
        return {"c": c, "da": da, "db": a.reshape(-1, case["k"]).t() @ dc.reshape(-1, case["n"])}
    if kind == "block":
        b, c, f, h, w = (case[x] for x in ("batch", "c", "f", "h", "w"))
        win = t["x"].view(b, c, h // 2, 2, w // 2, 2).permute(0, 1, 2, 4, 3, 5).reshape(b, c, h // 2, w // 2, 4)
        q = win.max(-1).values
        last = 3 - (win == q.unsqueeze(-1)).flip(-1).int().argmax(-1)  # ties go to the later element
        hot = torch.nn.functional.one_hot(last, 4)

        def back(v):
            return v.view(b, c, h // 2, w // 2, 2, 2).permute(0, 1, 2, 4, 3, 5).reshape(b, c, h, w).contiguous()

        pre = _conv_fwd(_h(q), _h(t["w"]), 1, 1) + t["b"].double().view(1, f, 1, 1)
        dq = _conv_dx(_h(t["dy"]), _h(t["w"]), 1, 1, h // 2, w // 2)
        return {"q": q.double(), "qmask": back(hot).int(), "y": pre.relu(), "ymask": _bits((pre > 0).float()), "dq": dq,
                "dx": back(hot.double() * dq.unsqueeze(-1)), "dw": _conv_dw(_h(t["dy"]), _h(q), 3, 1, 1), "db": t["dy"].double().sum((0, 2, 3))}
    k, s, p = case["k"], case["stride"], case["pad"]
    x, w, dy = _h(t["x"]), _h(t["w"]), _h(t["dy"])
    if kind == "convt":  # the adjoint of the convolution that has w as its weights
        ho, wo = _out_side(case)
        return {"y": _conv_dx(x, w, s, p, ho, wo), "dx": _conv_fwd(dy, w, s, p), "dw": _conv_dw(x, dy, k, s, p)}
    out = {"y": _conv_fwd(x, w, s, p), "dx": _conv_dx(dy, w, s, p, case["h"], case["w"]), "dw": _conv_dw(dy, x, k, s, p)}
    if case["bias"]:
        out["y"] += t["b"].double().view(1, -1, 1, 1)
        out["ymask"] = _bits((out["y"] > 0).float())
        out["y"] = out["y"].relu()
        out["db"] = t["dy"].double().sum((0, 2, 3))
    return out
