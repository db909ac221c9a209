"""The work that a user of this library has it do, as cases that can be timed and compared.

Every case goes through a public entry point: the C ABI of include/axis_hip.h through
axis_amd.hip (what a binding calls, layer by layer, on buffers it owns), or the C++ host layer
(axis_amd.host(): modules, tape, Trainer).  Buffers are torch tensors on the GPU; the handle's own
stream runs every launch.

Kinds, and what each stands for:

  mlp_step    one Trainer step (forward, backward, Adam) of a small MLP through the host layer, and
              the read-back of the loss and the updated weights: many short launches, where host
              work and latency count.
  head        a classifier head: Linear, mean softmax cross-entropy, its backward down to the
              features, through the C ABI.
  linear      one Linear layer, forward and backward (data, weight and bias gradient), on an fp32
              handle or (bf16) on a handle that rounds product operands to bf16.
  conv_block  Conv2d -> ReLU -> 2x2 max pool, forward and backward, channel-innermost input, or
              channel-major input without an input gradient when it is the first layer.
  conv        a plain Conv2d, forward and backward, of any kernel, size and channel count.
  cnn_step    a whole training step of the three-block CNN: logits, every gradient, Adam.
  muon        one Muon update of a weight matrix (momentum, five Newton-Schulz steps, apply).
  adam        one multi-tensor Adam update.
"""
import ctypes
import math

import numpy as np
import torch

import axis_amd
from axis_amd import hip

I64, I32, F32, VP = hip.I64, hip.I32, hip.F32, hip.VP
NS = (3.4445, -4.7750, 2.0315)
_devices = {}


def listed():
    return [
        # the smallest whole step: MLP 784-256-256-10, batch 128, through the Trainer
        {"name": "mlp_step_bs128", "kind": "mlp_step", "batch": 128, "inputs": 784, "hidden": 256, "classes": 10},
        # the CNN's classifier at its training batch: three short products and the loss
        {"name": "head_256x256x1000", "kind": "head", "rows": 256, "features": 256, "classes": 1000},
        # a layer of odd sizes, no extent a multiple of 4
        {"name": "linear_odd", "kind": "linear", "rows": 1531, "inputs": 1023, "outputs": 2049, "bf16": False},
        # the first layer of an MLP on flattened 28x28 images at a large batch
        {"name": "linear_8192x784x1024", "kind": "linear", "rows": 8192, "inputs": 784, "outputs": 1024, "bf16": False},
        # a wide hidden layer
        {"name": "linear_4096", "kind": "linear", "rows": 4096, "inputs": 4096, "outputs": 4096, "bf16": False},
        # the same layer on a bf16 device
        {"name": "linear_4096_bf16", "kind": "linear", "rows": 4096, "inputs": 4096, "outputs": 4096, "bf16": True},
        # the CNN's first block: 3 channels, channel-major images, no input gradient
        {"name": "conv_block_3x64", "kind": "conv_block", "batch": 256, "channels": 3, "outputs": 64, "size": 64},
        # the CNN's second block
        {"name": "conv_block_64x128", "kind": "conv_block", "batch": 256, "channels": 64, "outputs": 128, "size": 32},
        # a plain convolution of odd extents: 5x5 kernel, 21x19 images, 48 -> 80 channels
        {"name": "conv_odd", "kind": "conv", "batch": 50, "channels": 48, "outputs": 80, "height": 21, "width": 19,
         "kernel": 5, "padding": 2},
        # the whole training step of the three-block CNN (3-64-128-256, 64x64 images, 1000 classes)
        {"name": "cnn_step_bs256", "kind": "cnn_step", "batch": 256, "size": 64, "classes": 1000},
        # the wide MLP's first weight matrix under Muon
        {"name": "muon_4096x8192", "kind": "muon", "rows": 4096, "columns": 8192},
        # Adam over 16 tensors of 4,194,304 parameters
        {"name": "adam_16x4M", "kind": "adam", "tensors": 16, "length": 4194304},
    ]


def _log(rng, low, high):
    """A whole number, even over the logarithm of its range."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["mlp_step", "head", "linear", "linear", "linear", "conv_block", "conv_block", "conv", "cnn_step",
                       "muon", "adam"])

    def extent(low, high):
        # half of the extents are whole vectors and tiles, the others anything
        v = _log(rng, low, high)
        step = rng.choice([1, 1, 8, 32])
        return max(low, v // step * step) if step > 1 else v

    if kind == "mlp_step":
        return {"kind": kind, "batch": extent(16, 1024), "inputs": extent(32, 1024), "hidden": extent(32, 512),
                "classes": rng.randint(2, 100)}
    if kind == "head":
        return {"kind": kind, "rows": extent(16, 2048), "features": extent(32, 1024), "classes": extent(10, 1500)}
    if kind == "linear":
        return {"kind": kind, "rows": extent(64, 8192), "inputs": extent(48, 4096), "outputs": extent(16, 4096),
                "bf16": rng.random() < 0.3}
    if kind == "conv_block":
        if rng.random() < 0.3:
            return {"kind": kind, "batch": rng.randint(8, 256), "channels": rng.choice([1, 3]),
                    "outputs": rng.choice([16, 32, 64]), "size": rng.choice([28, 32, 48, 64])}
        size = rng.choice([8, 16, 16, 32, 32])
        channels, outputs = rng.choice([16, 32, 64, 96, 128]), rng.choice([32, 64, 96, 128, 192, 256])
        most = 256 * 32 * 32 * 64 * 128 // (size * size * channels * outputs)
        return {"kind": kind, "batch": rng.randint(4, max(8, min(512, most))), "channels": channels, "outputs": outputs,
                "size": size}
    if kind == "conv":
        kernel = rng.choice([1, 3, 3, 5])
        return {"kind": kind, "batch": rng.randint(2, 64), "channels": extent(4, 128), "outputs": extent(8, 160),
                "height": rng.randint(7, 33), "width": rng.randint(7, 33), "kernel": kernel, "padding": kernel // 2}
    if kind == "cnn_step":
        return {"kind": kind, "batch": rng.randint(16, 256), "size": rng.choice([16, 32, 64]),
                "classes": extent(10, 1000)}
    if kind == "muon":
        return {"kind": kind, "rows": extent(64, 4096), "columns": extent(64, 4096)}
    return {"kind": kind, "tensors": rng.randint(1, 16), "length": extent(100, 4194304)}


# ------------------------------------------------------------------ helpers


def _device(bf16=False):
    """One handle per operand mode for the life of the process, as a program keeps it."""
    if bf16 not in _devices:
        _devices[bf16] = hip.Device(0, bf16_matmul=bf16)
    return _devices[bf16]


def _p(t):
    return VP(t.data_ptr())


def _two(a, b):
    return (ctypes.c_int32 * 2)(a, b)


class _Gen:
    """Inputs on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 62) + 12345)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device="cuda", generator=self.g).mul_(std)

    def uniform(self, *shape):
        return torch.rand(*shape, device="cuda", generator=self.g)

    def activation(self, *shape):
        """What a ReLU layer hands on: about half zeros."""
        return self.normal(*shape).clamp_(min=0)

    def weight(self, fan_in, *shape):
        return self.normal(*shape, std=math.sqrt(2.0 / fan_in))

    def labels(self, rows, classes):
        at = torch.randint(classes, (rows,), device="cuda", generator=self.g)
        return torch.nn.functional.one_hot(at, classes).float()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


# ------------------------------------------------------------------ linear


def _linear_inputs(case, seed):
    g = _Gen(seed)
    m, k, n = case["rows"], case["inputs"], case["outputs"]
    return dict(x=g.activation(m, k), w=g.weight(k, k, n), b=g.normal(n, std=0.1), dy=g.normal(m, n, std=1.0 / m))


def _linear_prepare(case, seed):
    s = _linear_inputs(case, seed)
    m, k, n = case["rows"], case["inputs"], case["outputs"]
    s.update(dev=_device(case["bf16"]), m=m, k=k, n=n, y=_empty(m, n), dx=_empty(m, k), dw=_empty(k, n), db=_empty(n))
    return s


def _linear_run(s):
    call, m, k, n = s["dev"].call, I64(s["m"]), I64(s["k"]), I64(s["n"])
    x, w, b, dy = _p(s["x"]), _p(s["w"]), _p(s["b"]), _p(s["dy"])
    call("axis_matmul_bias", x, w, b, _p(s["y"]), I64(1), m, k, n)
    call("axis_matmul_left_backward", dy, w, _p(s["dx"]), I64(1), m, k, n)
    call("axis_matmul_right_backward", x, dy, _p(s["dw"]), I64(1), m, k, n)
    call("axis_bias_gradient", dy, None, None, _p(s["db"]), m, n)
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"], "db": s["db"]}


def _linear_exact(case, seed):
    s = _linear_inputs(case, seed)
    # a bf16 handle rounds the operands of its products, and nothing else
    op = (lambda t: t.bfloat16().double()) if case["bf16"] else (lambda t: t.double())
    x, w, dy = op(s["x"]), op(s["w"]), op(s["dy"])
    return {"y": x @ w + s["b"].double(), "dx": dy @ w.T, "dw": x.T @ dy, "db": s["dy"].double().sum(0)}


# ------------------------------------------------------------------ classifier head


def _head_inputs(case, seed):
    g = _Gen(seed)
    m, k, n = case["rows"], case["features"], case["classes"]
    return dict(x=g.activation(m, k), w=g.weight(k, k, n), b=g.normal(n, std=0.1), t=g.labels(m, n))


def _head_prepare(case, seed):
    s = _head_inputs(case, seed)
    m, k, n = case["rows"], case["features"], case["classes"]
    s.update(dev=_device(), m=m, k=k, n=n, one=torch.ones(1, device="cuda"), z=_empty(m, n), p=_empty(m, n),
             loss=_empty(m), mean=_empty(1), dz=_empty(m, n), db=_empty(n), dx=_empty(m, k), dw=_empty(k, n))
    return s


def _head_run(s):
    call, m, k, n = s["dev"].call, I64(s["m"]), I64(s["k"]), I64(s["n"])
    x, w, t, z, p, dz = _p(s["x"]), _p(s["w"]), _p(s["t"]), _p(s["z"]), _p(s["p"]), _p(s["dz"])
    share = F32(1.0 / s["m"])
    call("axis_matmul_bias", x, w, _p(s["b"]), z, I64(1), m, k, n)
    call("axis_softmax_cross_entropy", z, t, p, _p(s["loss"]), m, n)
    call("axis_reduce_middle", _p(s["loss"]), _p(s["mean"]), I64(1), m, I64(1), share)
    call("axis_categorical_cross_entropy_backward_mean", _p(s["one"]), share, p, t, dz, _p(s["db"]), m, n)
    call("axis_matmul_left_backward", dz, w, _p(s["dx"]), I64(1), m, k, n)
    call("axis_matmul_right_backward", x, dz, _p(s["dw"]), I64(1), m, k, n)
    return {"z": s["z"], "p": s["p"], "loss": s["loss"], "mean": s["mean"], "dz": s["dz"], "db": s["db"], "dx": s["dx"],
            "dw": s["dw"]}


def _head64(x, w, b, t):
    z = x @ w + b
    logs = z - torch.logsumexp(z, 1, keepdim=True)
    p = logs.exp()
    loss = -(logs * t).sum(1)
    dz = (p - t) / x.shape[0]
    return {"z": z, "p": p, "loss": loss, "mean": loss.mean().reshape(1), "dz": dz, "db": dz.sum(0), "dx": dz @ w.T,
            "dw": x.T @ dz}


def _head_exact(case, seed):
    s = _head_inputs(case, seed)
    return _head64(s["x"].double(), s["w"].double(), s["b"].double(), s["t"].double())


# ------------------------------------------------------------------ convolutions
#
# Tensors are channel-innermost [batch, height, width, channels]; weights [(channel, ky, kx), out].


def _taps64(x, w, kernel, padding):
    """The stride-1 convolution of x [b, h, w, c] in 64 bits, tap by tap."""
    b, h, wd, c = x.shape
    n = w.shape[1]
    w4 = w.reshape(c, kernel, kernel, n)
    xp = torch.nn.functional.pad(x, (0, 0, padding, padding, padding, padding))
    oh, ow = h + 2 * padding - kernel + 1, wd + 2 * padding - kernel + 1
    y = torch.zeros(b * oh * ow, n, device=x.device, dtype=torch.float64)
    for ky in range(kernel):
        for kx in range(kernel):
            y += xp[:, ky:ky + oh, kx:kx + ow].reshape(-1, c) @ w4[:, ky, kx]
    return y.reshape(b, oh, ow, n)


def _taps64_backward(x, w, dy, kernel, padding, data=True):
    b, h, wd, c = x.shape
    n = w.shape[1]
    w4 = w.reshape(c, kernel, kernel, n)
    xp = torch.nn.functional.pad(x, (0, 0, padding, padding, padding, padding))
    oh, ow = dy.shape[1:3]
    g = dy.reshape(-1, n)
    dw = torch.zeros_like(w4)
    dx = torch.zeros_like(xp) if data else None
    for ky in range(kernel):
        for kx in range(kernel):
            dw[:, ky, kx] = xp[:, ky:ky + oh, kx:kx + ow].reshape(-1, c).T @ g
            if data:
                dx[:, ky:ky + oh, kx:kx + ow] += (g @ w4[:, ky, kx].T).reshape(b, oh, ow, c)
    return dw.reshape(w.shape), dx[:, padding:padding + h, padding:padding + wd] if data else None


def _unpool(g, pooled, argmax):
    """The pre-activation gradient of ReLU -> 2x2 max pool: g at each window's winner where the pooled value is > 0."""
    b, ph, pw, n = g.shape
    g = torch.where(pooled > 0, g, torch.zeros_like(g))
    out = torch.zeros(b, ph, 2, pw, 2, n, device=g.device, dtype=g.dtype)
    for ky in range(2):
        for kx in range(2):
            out[:, :, ky, :, kx] = torch.where(argmax == 2 * ky + kx, g, torch.zeros_like(g))
    return out.reshape(b, 2 * ph, 2 * pw, n)


def _first(case):
    """A first layer: few channels, images as they are loaded (channel-major), no input gradient."""
    return case["channels"] <= 3


def _block_inputs(case, seed):
    g = _Gen(seed)
    b, c, n, size = case["batch"], case["channels"], case["outputs"], case["size"]
    x = g.uniform(b, c, size, size) if _first(case) else g.activation(b, size, size, c)
    # a forward pass's saved values: the pooled outputs of ReLU and the winners (0 where nothing is positive)
    pooled = g.normal(b, size // 2, size // 2, n).add_(0.8).clamp_(min=0)
    winner = torch.randint(4, pooled.shape, device="cuda", generator=g.g, dtype=torch.uint8)
    winner *= pooled > 0
    return dict(x=x, w=g.weight(9 * c, 9 * c, n), b=g.normal(n, std=0.1), pooled=pooled, winner=winner,
                g=g.normal(*pooled.shape, std=1.0 / pooled[..., 0].numel()))


def _block_prepare(case, seed):
    s = _block_inputs(case, seed)
    b, c, n, size = case["batch"], case["channels"], case["outputs"], case["size"]
    s.update(dev=_device(), case=case, y=torch.empty_like(s["pooled"]), at=torch.empty_like(s["winner"]),
             dw=torch.empty_like(s["w"]), db=torch.empty_like(s["b"]))
    s["strides"] = (ctypes.c_int64 * 4)(c * size * size, size * size, size, 1) if _first(case) else None
    if not _first(case):
        s.update(pre=_empty(b, size, size, n), dx=torch.empty_like(s["x"]))
    return s


def _block_run(s):
    case, call = s["case"], s["dev"].call
    b, c, n, size = I64(case["batch"]), I32(case["channels"]), I32(case["outputs"]), I32(case["size"])
    x, w, st = _p(s["x"]), _p(s["w"]), s["strides"]
    k, one, pool = _two(3, 3), _two(1, 1), _two(2, 2)
    call("axis_conv2d_relu_pool_forward", x, st, w, _p(s["b"]), _p(s["y"]), _p(s["at"]), b, size, size, c, n, k, one, one,
         pool)
    out = {"y": s["y"], "at": s["at"], "dw": s["dw"], "db": s["db"]}
    saved = _p(s["g"]), _p(s["pooled"]), _p(s["winner"])
    if s["strides"] is not None:
        call("axis_conv2d_relu_pool_backward_weight", x, st, *saved, _p(s["dw"]), _p(s["db"]), b, size, size, c, n, k, one,
             one, pool)
        return out
    pre = _p(s["pre"])
    call("axis_relu_pool_backward", *saved, pre, _p(s["db"]), b, size, size, n, pool)
    call("axis_conv2d_backward_data", pre, w, _p(s["dx"]), b, size, size, c, n, k, one, one)
    call("axis_conv2d_backward_weight", x, None, pre, _p(s["dw"]), b, size, size, c, n, k, one, one)
    return dict(out, pre=s["pre"], dx=s["dx"])


def _block_exact(case, seed):
    s = _block_inputs(case, seed)
    x = (s["x"].permute(0, 2, 3, 1) if _first(case) else s["x"]).double()
    w = s["w"].double()
    z = _taps64(x, w, 3, 1) + s["b"].double()
    y = torch.nn.functional.max_pool2d(z.clamp_(min=0).permute(0, 3, 1, 2), 2).permute(0, 2, 3, 1)
    pre = _unpool(s["g"].double(), s["pooled"], s["winner"])
    dw, dx = _taps64_backward(x, w, pre, 3, 1, data=not _first(case))
    # the winners are whole numbers that a tie may move: no 64-bit value
    out = {"y": y.contiguous(), "at": None, "dw": dw, "db": pre.sum((0, 1, 2))}
    return out if _first(case) else dict(out, pre=pre, dx=dx.contiguous())


def _conv_inputs(case, seed):
    g = _Gen(seed)
    b, c, n, h, w, k, p = (case[x] for x in ("batch", "channels", "outputs", "height", "width", "kernel", "padding"))
    oh, ow = h + 2 * p - k + 1, w + 2 * p - k + 1
    return dict(x=g.activation(b, h, w, c), w=g.weight(k * k * c, k * k * c, n), b=g.normal(n, std=0.1),
                dy=g.normal(b, oh, ow, n, std=1.0 / (b * oh * ow)))


def _conv_prepare(case, seed):
    s = _conv_inputs(case, seed)
    s.update(dev=_device(), case=case, y=torch.empty_like(s["dy"]), dx=torch.empty_like(s["x"]),
             dw=torch.empty_like(s["w"]), db=torch.empty_like(s["b"]))
    return s


def _conv_run(s):
    case, call = s["case"], s["dev"].call
    k, one, p = _two(case["kernel"], case["kernel"]), _two(1, 1), _two(case["padding"], case["padding"])
    shape = (I64(case["batch"]), I32(case["height"]), I32(case["width"]), I32(case["channels"]), I32(case["outputs"]), k, one,
             p)
    x, w, dy = _p(s["x"]), _p(s["w"]), _p(s["dy"])
    call("axis_conv2d_forward", x, None, w, _p(s["b"]), _p(s["y"]), *shape)
    n = case["outputs"]
    call("axis_bias_gradient", dy, None, None, _p(s["db"]), I64(s["dy"].numel() // n), I64(n))
    call("axis_conv2d_backward_data", dy, w, _p(s["dx"]), *shape)
    call("axis_conv2d_backward_weight", x, None, dy, _p(s["dw"]), *shape)
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"], "db": s["db"]}


def _conv_exact(case, seed):
    s = _conv_inputs(case, seed)
    x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
    dw, dx = _taps64_backward(x, w, dy, case["kernel"], case["padding"])
    return {"y": _taps64(x, w, case["kernel"], case["padding"]) + s["b"].double(), "dx": dx.contiguous(), "dw": dw,
            "db": dy.sum((0, 1, 2))}


# ------------------------------------------------------------------ the CNN's training step

CHANNELS = (3, 64, 128, 256)
ADAM = (1e-3, 0.9, 0.999, 1e-8)
ADAM_STEP = 101  # warm moments, as in the middle of a run


def _cnn_inputs(case, seed):
    g = _Gen(seed)
    b, size, classes = case["batch"], case["size"], case["classes"]
    params = []
    for j in range(3):
        params += [g.weight(9 * CHANNELS[j], 9 * CHANNELS[j], CHANNELS[j + 1]), g.normal(CHANNELS[j + 1], std=0.05)]
    params += [g.weight(CHANNELS[3], CHANNELS[3], classes), g.normal(classes, std=0.05)]
    first = [g.normal(*p.shape, std=1e-3) for p in params]
    second = [g.normal(*p.shape, std=1e-3).square_().add_(1e-8) for p in params]
    return dict(x=g.uniform(b, 3, size, size), t=g.labels(b, classes), params=params, first=first, second=second)


def _adam_tensors(params, grads, first, second):
    return (hip.AdamTensor * len(params))(*[
        hip.AdamTensor(p.data_ptr(), g.data_ptr(), m.data_ptr(), v.data_ptr(), None, p.numel())
        for p, g, m, v in zip(params, grads, first, second)])


def _adam_call(dev, tensors, step):
    lr, b1, b2, eps = ADAM
    dev.call("axis_adam_multi", tensors, I32(len(tensors)), F32(lr), F32(b1), F32(b2), F32(1 - b1 ** step),
             F32(1 - b2 ** step), F32(eps), F32(0.0))


def _cnn_prepare(case, seed):
    s = _cnn_inputs(case, seed)
    b, size, classes = case["batch"], case["size"], case["classes"]
    s.update(dev=_device(), case=case, grads=[torch.empty_like(p) for p in s["params"]], one=torch.ones(1, device="cuda"))
    s["tensors"] = _adam_tensors(s["params"], s["grads"], s["first"], s["second"])
    for j in range(3):
        hw, n = size >> j, CHANNELS[j + 1]
        s["y%d" % j], s["at%d" % j] = _empty(b, hw // 2, hw // 2, n), _empty(b, hw // 2, hw // 2, n, dtype=torch.uint8)
        if j:
            s["pre%d" % j], s["dx%d" % j] = _empty(b, hw, hw, n), _empty(b, hw, hw, CHANNELS[j])
    d = CHANNELS[3]
    s.update(mean=_empty(b, d), z=_empty(b, classes), p=_empty(b, classes), rows=_empty(b), loss=_empty(1),
             dz=_empty(b, classes), dmean=_empty(b, d))
    return s


def _cnn_run(s):
    case, call, params, grads = s["case"], s["dev"].call, s["params"], s["grads"]
    batch, size, classes = case["batch"], case["size"], case["classes"]
    b, d, n = I64(batch), I64(CHANNELS[3]), I64(classes)
    k, one, pool = _two(3, 3), _two(1, 1), _two(2, 2)
    strides = (ctypes.c_int64 * 4)(3 * size * size, size * size, size, 1)
    shape = [(b, I32(size >> j), I32(size >> j), I32(CHANNELS[j]), I32(CHANNELS[j + 1])) for j in range(3)]
    x = [s["x"], s["y0"], s["y1"]]
    for j in range(3):
        call("axis_conv2d_relu_pool_forward", _p(x[j]), None if j else strides, _p(params[2 * j]), _p(params[2 * j + 1]),
             _p(s["y%d" % j]), _p(s["at%d" % j]), *shape[j], k, one, one, pool)
    last = size >> 3
    call("axis_reduce_middle", _p(s["y2"]), _p(s["mean"]), b, I64(last * last), d, F32(1.0 / (last * last)))
    share = F32(1.0 / batch)
    call("axis_matmul_bias", _p(s["mean"]), _p(params[6]), _p(params[7]), _p(s["z"]), I64(1), b, d, n)
    call("axis_softmax_cross_entropy", _p(s["z"]), _p(s["t"]), _p(s["p"]), _p(s["rows"]), b, n)
    call("axis_reduce_middle", _p(s["rows"]), _p(s["loss"]), I64(1), b, I64(1), share)
    # backward, as the tape runs it: the last sums of the weight and bias gradients in one launch
    call("axis_finish_defer", I32(1))
    call("axis_categorical_cross_entropy_backward_mean", _p(s["one"]), share, _p(s["p"]), _p(s["t"]), _p(s["dz"]),
         _p(grads[7]), b, n)
    call("axis_matmul_left_backward", _p(s["dz"]), _p(params[6]), _p(s["dmean"]), I64(1), b, d, n)
    call("axis_matmul_right_backward", _p(s["mean"]), _p(s["dz"]), _p(grads[6]), I64(1), b, d, n)
    for j in (2, 1):
        hw, c = I32(size >> j), I32(CHANNELS[j + 1])
        saved = _p(s["y%d" % j]), _p(s["at%d" % j]), _p(s["pre%d" % j]), _p(grads[2 * j + 1]), b, hw, hw, c, pool
        if j == 2:
            call("axis_relu_pool_backward_mean", _p(s["dmean"]), F32(1.0 / (last * last)), *saved)
        else:
            call("axis_relu_pool_backward", _p(s["dx2"]), *saved)
        call("axis_conv2d_backward_data", _p(s["pre%d" % j]), _p(params[2 * j]), _p(s["dx%d" % j]), *shape[j], k, one, one)
        call("axis_conv2d_backward_weight", _p(x[j]), None, _p(s["pre%d" % j]), _p(grads[2 * j]), *shape[j], k, one, one)
    call("axis_conv2d_relu_pool_backward_weight", _p(x[0]), strides, _p(s["dx1"]), _p(s["y0"]), _p(s["at0"]), _p(grads[0]),
         _p(grads[1]), *shape[0], k, one, one, pool)
    call("axis_finish_defer", I32(0))
    _adam_call(s["dev"], s["tensors"], ADAM_STEP)
    return {"z": s["z"], "loss": s["loss"], "grads": list(grads), "params": list(params), "first": list(s["first"]),
            "second": list(s["second"])}


def _cnn_exact(case, seed):
    s = _cnn_inputs(case, seed)
    p = [t.double() for t in s["params"]]
    x = s["x"].permute(0, 2, 3, 1).double()
    for j in range(3):
        y = (_taps64(x, p[2 * j], 3, 1) + p[2 * j + 1]).clamp_(min=0)
        x = torch.nn.functional.max_pool2d(y.permute(0, 3, 1, 2), 2).permute(0, 2, 3, 1).contiguous()
    head = _head64(x.mean((1, 2)), p[6], p[7], s["t"].double())
    # The convolutions' gradients hang on each window's winner, and two values that agree to rounding may each win
    # one: no 64-bit value to hold them to, nor the updates made from them.
    none = [None] * 6
    grads = none + [head["dw"], head["db"]]
    lr, b1, b2, eps = ADAM
    first = none + [b1 * s["first"][i].double() + (1 - b1) * grads[i] for i in (6, 7)]
    second = none + [b2 * s["second"][i].double() + (1 - b2) * grads[i] ** 2 for i in (6, 7)]
    params = none + [p[i] - lr * (first[i] / (1 - b1 ** ADAM_STEP)) / ((second[i] / (1 - b2 ** ADAM_STEP)).sqrt() + eps)
                     for i in (6, 7)]
    return {"z": head["z"], "loss": head["mean"], "grads": grads, "params": params, "first": first, "second": second}


# ------------------------------------------------------------------ optimizers


def _adam_inputs(case, seed):
    g = _Gen(seed)
    n = case["length"]
    tensors = range(case["tensors"])
    return dict(params=[g.normal(n, std=0.02) for _ in tensors], grads=[g.normal(n, std=1e-3) for _ in tensors],
                first=[g.normal(n, std=3e-4) for _ in tensors],
                second=[g.normal(n, std=1e-3).square_().add_(1e-10) for _ in tensors])


def _adam_prepare(case, seed):
    s = _adam_inputs(case, seed)
    s["tensors"] = _adam_tensors(s["params"], s["grads"], s["first"], s["second"])
    return dict(s, dev=_device())


def _adam_run(s):
    _adam_call(s["dev"], s["tensors"], ADAM_STEP)
    return {"params": s["params"], "first": s["first"], "second": s["second"]}


def _adam_exact(case, seed):
    s = _adam_inputs(case, seed)
    lr, b1, b2, eps = ADAM
    out = {"params": [], "first": [], "second": []}
    for p, g, m, v in zip(s["params"], s["grads"], s["first"], s["second"]):
        g = g.double()
        m, v = b1 * m.double() + (1 - b1) * g, b2 * v.double() + (1 - b2) * g * g
        out["params"].append(p.double() - lr * (m / (1 - b1 ** ADAM_STEP)) / ((v / (1 - b2 ** ADAM_STEP)).sqrt() + eps))
        out["first"].append(m)
        out["second"].append(v)
    return out


def _muon_inputs(case, seed):
    g = _Gen(seed)
    shape = (case["rows"], case["columns"])
    return dict(w=g.weight(shape[0], *shape), g=g.normal(*shape, std=1e-3), m=g.normal(*shape, std=1e-3))


def _muon_prepare(case, seed):
    s = _muon_inputs(case, seed)
    r, c = case["rows"], case["columns"]
    small = min(r, c)
    s.update(dev=_device(), r=r, c=c, next=_empty(r, c), dir=_empty(r, c), out=_empty(r, c), x=[_empty(r, c), _empty(r, c)],
             gram=_empty(small, small), b=_empty(small, small), sq=_empty(1), inv=_empty(1))
    return s


def _muon_run(s):
    call, r, c = s["dev"].call, s["r"], s["c"]
    small, n = min(r, c), I64(r * c)
    a, b, cc = (F32(v) for v in NS)
    mu = F32(0.95)
    call("axis_muon_momentum", _p(s["g"]), _p(s["m"]), _p(s["next"]), _p(s["dir"]), mu, I32(1), n)
    call("axis_sum_squares", _p(s["dir"]), n, _p(s["sq"]))
    call("axis_inverse_sqrt", _p(s["sq"]), F32(1e-14), _p(s["inv"]), I64(1))
    x, y = s["x"]
    call("axis_multiply_scalar", _p(s["dir"]), _p(s["inv"]), _p(x), n)
    gram, bb, one, sm = _p(s["gram"]), _p(s["b"]), I64(1), I64(small)
    for _ in range(5):
        if r <= c:
            call("axis_matmul_left_backward", _p(x), _p(x), gram, one, sm, sm, I64(c))
        else:
            call("axis_matmul_right_backward", _p(x), _p(x), gram, one, I64(r), sm, sm)
        call("axis_matmul_axpby", gram, gram, gram, bb, one, sm, sm, sm, cc, b)
        if r <= c:
            call("axis_matmul_axpby", bb, _p(x), _p(x), _p(y), one, sm, sm, I64(c), F32(1.0), a)
        else:
            call("axis_matmul_axpby", _p(x), bb, _p(x), _p(y), one, I64(r), sm, sm, F32(1.0), a)
        x, y = y, x
    scale = math.sqrt(max(c / r, 1.0))
    call("axis_muon_apply", _p(s["w"]), _p(x), _p(s["out"]), F32(1.0 - 0.02 * 0.01), F32(0.02 * scale), n)
    return {"weight": s["out"], "momentum": s["next"], "orthogonal": x}


def _muon_exact(case, seed):
    s = _muon_inputs(case, seed)
    a, b, c = NS
    g = s["g"].double()
    m = 0.95 * s["m"].double() + 0.05 * g
    x = 0.05 * g + 0.95 * m
    x = x / (x.square().sum() + 1e-14).sqrt()
    flip = case["rows"] > case["columns"]
    x = x.T.contiguous() if flip else x
    for _ in range(5):
        gram = x @ x.T
        x = a * x + (b * gram + c * (gram @ gram)) @ x
    x = x.T.contiguous() if flip else x
    scale = math.sqrt(max(case["columns"] / case["rows"], 1.0))
    return {"weight": s["w"].double() * (1.0 - 0.02 * 0.01) - 0.02 * scale * x, "momentum": m, "orthogonal": x}


# ------------------------------------------------------------------ MLP step through the host layer


def _mlp_inputs(case, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    sizes = (case["inputs"], case["hidden"], case["hidden"], case["classes"])
    weights = [rng.standard_normal((sizes[j], sizes[j + 1])).astype(np.float32) * np.float32(math.sqrt(2.0 / sizes[j]))
               for j in range(3)]
    biases = [rng.standard_normal(sizes[j + 1]).astype(np.float32) * np.float32(0.05) for j in range(3)]
    x = rng.random_sample((case["batch"], sizes[0])).astype(np.float32)
    t = np.eye(sizes[3], dtype=np.float32)[rng.randint(0, sizes[3], case["batch"])]
    return sizes, weights, biases, x, t


def _mlp_prepare(case, seed):
    ax = axis_amd.host()
    if "host" not in _devices:
        _devices["host"] = ax.Device.hip(0)
    device = _devices["host"]
    sizes, weights, biases, x, t = _mlp_inputs(case, seed)
    bt, f = ax.Axis("batch"), [ax.Axis("f%d" % j) for j in range(4)]
    layers = []
    for j in range(3):
        layers.append(ax.Linear(f[j], f[j + 1].of(sizes[j + 1])))
        if j < 2:
            layers.append(ax.ReLU())
    model = ax.Sequential(layers)
    model.build(ax.Shape([bt.of(case["batch"]), f[0].of(sizes[0])]), device, 1)
    params = []
    for j in range(3):
        for name, value in (("weight", weights[j]), ("bias", biases[j])):
            params.append(model.parameter("%d.%s" % (2 * j, name)))
            params[-1].set_values(value.reshape(-1))
    xt = ax.Tensor.from_slice(x.reshape(-1), [bt.of(case["batch"]), f[0].of(sizes[0])], device)
    tt = ax.Tensor.from_slice(t.reshape(-1), [bt.of(case["batch"]), f[3].of(sizes[3])], device)
    trainer = ax.Trainer(ax.Adam(ADAM[0]))

    def loss(m):
        return m.forward(xt).categorical_cross_entropy_with_logits(tt, f[3]).mean([bt])

    return dict(model=model, params=params, trainer=trainer, loss=loss)


def _mlp_run(s):
    _, loss = s["trainer"].step(s["model"], s["loss"])
    return {"loss": loss.item(), "params": [p.tensor().to_vec() for p in s["params"]]}


def _mlp_exact(case, seed):
    sizes, weights, biases, x, t = _mlp_inputs(case, seed)
    p = [torch.from_numpy(v).double().requires_grad_() for w, b in zip(weights, biases) for v in (w, b)]
    h = torch.from_numpy(x).double()
    for j in range(3):
        h = h @ p[2 * j] + p[2 * j + 1]
        if j < 2:
            h = h.clamp(min=0)
    loss = -(torch.log_softmax(h, 1) * torch.from_numpy(t).double()).sum(1).mean()
    loss.backward()
    lr, _, _, eps = ADAM
    # Adam's first step from zero moments: lr * g / (|g| + eps)
    return {"loss": loss.detach(),
            "params": [(v.detach() - lr * v.grad / (v.grad.abs() + eps)).reshape(-1) for v in p]}


# ------------------------------------------------------------------ the interface

_KINDS = {
    "mlp_step": (_mlp_prepare, _mlp_run, _mlp_exact),
    "head": (_head_prepare, _head_run, _head_exact),
    "linear": (_linear_prepare, _linear_run, _linear_exact),
    "conv_block": (_block_prepare, _block_run, _block_exact),
    "conv": (_conv_prepare, _conv_run, _conv_exact),
    "cnn_step": (_cnn_prepare, _cnn_run, _cnn_exact),
    "muon": (_muon_prepare, _muon_run, _muon_exact),
    "adam": (_adam_prepare, _adam_run, _adam_exact),
}


def prepare(case, seed):
    return {"kind": case["kind"], "state": _KINDS[case["kind"]][0](case, seed)}


def run(state):
    return _KINDS[state["kind"]][1](state["state"])


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def _linear_work(m, k, n):
    """Forward, data, weight and bias gradient: x, w, b, dy read once, y, dx, dw, db written once."""
    return {"bytes": 4.0 * 2 * (m * k + k * n + m * n + n), "flops": 6.0 * m * k * n}


def _block_work(b, c, n, size, first):
    pixels, windows = b * size * size, b * size * size / 4
    flops = 2.0 * pixels * 9 * c * n * (2 if first else 3)
    # x, w, bias and the saved g, pooled, winner read; pooled, winner, dw, db (and pre, dx) written
    size4 = 4.0 * (pixels * c + 2 * (9 * c * n + n)) + windows * n * (9 + 5)
    return {"bytes": size4 + (0 if first else 4.0 * pixels * (n + c)), "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["rows"], case["inputs"], case["outputs"])
    if kind == "head":
        m, k, n = case["rows"], case["features"], case["classes"]
        # x, w, b, t read; logits, probabilities, dz, dx, dw, db, loss written
        return {"bytes": 4.0 * (2 * m * k + 2 * k * n + 4 * m * n + 2 * n + m), "flops": 6.0 * m * k * n}
    if kind == "mlp_step":
        i, h, c, b = case["inputs"], case["hidden"], case["classes"], case["batch"]
        weights = i * h + h * h + h * c + 2 * h + c
        return {"bytes": 28.0 * weights + 4.0 * b * (i + c), "flops": 6.0 * b * weights - 2.0 * b * i * h}
    if kind == "conv_block":
        return _block_work(case["batch"], case["channels"], case["outputs"], case["size"], _first(case))
    if kind == "conv":
        b, c, n, k, p = (case[x] for x in ("batch", "channels", "outputs", "kernel", "padding"))
        pixels = b * case["height"] * case["width"]
        outs = b * (case["height"] + 2 * p - k + 1) * (case["width"] + 2 * p - k + 1)
        return {"bytes": 8.0 * (pixels * c + outs * n + k * k * c * n + n), "flops": 6.0 * outs * k * k * c * n}
    if kind == "cnn_step":
        b, size, classes = case["batch"], case["size"], case["classes"]
        flops, weights = 6.0 * b * CHANNELS[3] * classes, CHANNELS[3] * classes + classes
        moved = 4.0 * b * (3 * size * size + classes)  # images and labels
        for j in range(3):
            w = _block_work(b, CHANNELS[j], CHANNELS[j + 1], size >> j, j == 0)
            flops += w["flops"]
            weights += 9 * CHANNELS[j] * CHANNELS[j + 1] + CHANNELS[j + 1]
            # each pooled output and winner written, then read again by the backward
            moved += 2 * 5.0 * b * (size >> j) ** 2 / 4 * CHANNELS[j + 1]
        return {"bytes": moved + 28.0 * weights, "flops": flops}
    if kind == "muon":
        s, l = sorted((case["rows"], case["columns"]))
        # w, g, momentum read; weight, momentum, orthogonal written
        return {"bytes": 24.0 * s * l, "flops": 5 * (4.0 * s * s * l + 2.0 * s * s * s)}
    return {"bytes": 28.0 * case["tensors"] * case["length"], "flops": 12.0 * case["tensors"] * case["length"]}


def tolerance(case):
    """About four times what an fp32 result was measured to lie from the 64-bit one, or to move when its inputs move by
    a rounding, whichever is more."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 2e-6 if case["bf16"] else 5e-6}
    if kind == "cnn_step":
        # a whole call: a rounding moves single winners of the pools, and each takes a gradient term with it
        return {"rel": 4e-4, "max": 0.01}
    if kind == "muon":
        # five Newton-Schulz steps, each of which can amplify a rounding threefold
        return {"rel": 3e-5}
    if kind == "mlp_step":
        # Adam's first step moves an element whose gradient is within rounding of zero by up to the learning rate
        return {"rel": 2e-6, "max": 0.05}
    if kind == "adam":
        return {"rel": 1e-6}
    # one layer or block; of its winners (conv_block), those whose two best values agree to rounding may differ
    return {"rel": 2e-6, "differ": 1e-5 if kind == "conv_block" else 0.0}
