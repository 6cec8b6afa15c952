"""The work that users of this library have it do, as cases to be measured.

Four kinds of case, all through the public entry points (``singa_amd.workloads`` / ``singa_wrap`` / ``opt``):

* ``train``  -- a network of ``workloads``: a whole training step (forward, backward, SGD-momentum update) or, with
  ``mode`` "backward", the backward pass + update on activations that are already there (what ``bench.py`` times).
  ``tape`` "fused" is the tape with the library's fused calls; "reference" is one call per tensor op on one stream
  with the update op by op, what an unchanged autograd / optimizer issues.
* ``conv``   -- one convolution layer: forward, data, weight and (fp32 with bias) bias gradient.
* ``norm``   -- BatchNorm + ReLU, and a pooling layer of the same size, forward and backward.
* ``linear`` -- one dense layer, forward and backward.

``listed`` names twelve of them, ``draw`` picks others of the same ranges.
"""
import numpy as np
import torch

from singa_amd import singa_wrap as singa
from singa_amd import workloads

TORCH_TYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SINGA_TYPE = {"f32": singa.kFloat32, "f16": singa.kFloat16, "bf16": singa.kBFloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
LR, MOMENTUM = 1e-3, 0.9   # a small rate: a state is stepped hundreds of times on one batch and has to stay in range


def listed():
    return [
        # the MLP of examples/mlp at its batch: a step of a dozen short kernels, launches and host work count
        {"name": "mlp_step_b128", "kind": "train", "net": "mlp", "storage": "f32", "batch": 128, "width": 784, "hidden": 1000,
         "classes": 10, "tape": "fused", "mode": "step"},
        # the small CIFAR network (5x5 convolutions with bias, 2x2 pooling, one dense layer) at its batch
        {"name": "cnn_step_b128", "kind": "train", "net": "cnn", "storage": "f32", "batch": 128, "image": 32, "c1": 32, "c2": 64,
         "classes": 10, "tape": "fused", "mode": "step"},
        # ResNet-18 at the benchmark's batch: a whole training step in fp32
        {"name": "resnet18_step_f32_b64", "kind": "train", "net": "resnet18", "storage": "f32", "batch": 64, "image": 224,
         "classes": 1000, "tape": "fused", "mode": "step"},
        # the benchmark's own timed region: backward + update on resident activations
        {"name": "resnet18_backward_f32_b64", "kind": "train", "net": "resnet18", "storage": "f32", "batch": 64, "image": 224,
         "classes": 1000, "tape": "fused", "mode": "backward"},
        # a small odd batch of smaller images (planes of 80, 40, 20, 10, 5) through unchanged host code: one call per op
        {"name": "resnet18_reference_tape_b13", "kind": "train", "net": "resnet18", "storage": "f32", "batch": 13, "image": 160,
         "classes": 100, "tape": "reference", "mode": "step"},
        # ResNet-50 in mixed precision at the benchmark's batch: the largest
        {"name": "resnet50_step_f16_b128", "kind": "train", "net": "resnet50", "storage": "f16", "batch": 128, "image": 224,
         "classes": 1000, "tape": "fused", "mode": "step"},
        # the same network in bfloat16 on a small odd batch of 192-pixel images (planes of 96, 48, 24, 12, 6)
        {"name": "resnet50_step_bf16_b21", "kind": "train", "net": "resnet50", "storage": "bf16", "batch": 21, "image": 192,
         "classes": 1000, "tape": "fused", "mode": "step"},
        # the single convolution layer of the benchmark configurations, with bias
        {"name": "conv3x3_f32", "kind": "conv", "storage": "f32", "n": 64, "c": 64, "h": 56, "w": 56, "k": 64, "r": 3, "stride": 1,
         "pad": 1, "groups": 1, "bias": True},
        # a layer whose every size is ragged: channels that fill no tile, odd planes, an odd batch
        {"name": "conv3x3_bf16_ragged", "kind": "conv", "storage": "bf16", "n": 37, "c": 72, "h": 31, "w": 45, "k": 136, "r": 3,
         "stride": 1, "pad": 1, "groups": 1, "bias": False},
        # the depthwise half of a separable convolution (the handle's `groups`)
        {"name": "conv3x3_depthwise_f32", "kind": "conv", "storage": "f32", "n": 32, "c": 96, "h": 28, "w": 28, "k": 96, "r": 3,
         "stride": 1, "pad": 1, "groups": 96, "bias": False},
        # BatchNorm + ReLU and the residual networks' max pooling on odd planes
        {"name": "norm_pool_bf16_ragged", "kind": "norm", "storage": "bf16", "n": 50, "c": 72, "h": 57, "w": 43, "pool": 3,
         "pool_stride": 2, "pool_pad": 1, "max": True},
        # the classifier of a pure half model
        {"name": "linear_f16_b256", "kind": "linear", "storage": "f16", "batch": 256, "width": 2048, "out": 1000},
    ]


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _chosen(rng, options):
    """(value, weight) pairs -> a value."""
    return rng.choices([v for v, _ in options], [w for _, w in options])[0]


def _draw_train(rng):
    net = _chosen(rng, [("mlp", 2), ("cnn", 2), ("resnet18", 3), ("resnet50", 3)])
    case = {"kind": "train", "net": net, "storage": "f32", "tape": _chosen(rng, [("fused", 7), ("reference", 3)]),
            "mode": _chosen(rng, [("step", 7), ("backward", 3)])}
    if net == "mlp":
        return dict(case, batch=_log_int(rng, 1, 1024), width=_log_int(rng, 32, 4096), hidden=_log_int(rng, 32, 4096),
                    classes=_log_int(rng, 2, 1000))
    if net == "cnn":
        return dict(case, batch=_log_int(rng, 1, 512), image=4 * rng.randint(5, 16), c1=rng.choice([8, 16, 24, 32, 48]),
                    c2=rng.choice([16, 32, 64, 80]), classes=_log_int(rng, 2, 100))
    if net == "resnet50":
        case["storage"] = rng.choice(["f16", "bf16"])
    image = 32 * rng.randint(4, 8)
    # at most the pixels of the listed batches of 64 and 128 (call by call a step takes longer: three quarters of them); at
    # least eight images, so that BatchNorm has something to average
    most = {"resnet18": 64, "resnet50": 128}[net] * (224.0 / image) ** 2
    most = int(most * (0.75 if case["tape"] == "reference" else 1))
    return dict(case, batch=_log_int(rng, 8, min(256, most)), image=image, classes=_log_int(rng, 10, 1000))


def _draw_conv(rng):
    storage = _chosen(rng, [("f32", 4), ("f16", 3), ("bf16", 3)])
    r = _chosen(rng, [(1, 3), (3, 5), (5, 1), (7, 1)])
    stride = _chosen(rng, [(1, 3), (2, 1)])
    grouping = _chosen(rng, [("dense", 8), ("grouped", 1), ("depthwise", 1)])
    while True:
        n, h = _log_int(rng, 1, 128), _log_int(rng, 7, 112)
        w = max(7, min(112, int(h * rng.uniform(0.7, 1.4))))
        if grouping == "dense":
            c, k, groups = _log_int(rng, 3, 1024), _log_int(rng, 8, 1024), 1
        elif grouping == "grouped":
            groups = rng.choice([2, 4, 8])
            c, k = groups * _log_int(rng, 4, 64), groups * _log_int(rng, 4, 64)
        else:
            c = k = groups = _log_int(rng, 8, 96)
        p, q = (h + 2 * (r // 2) - r) // stride + 1, (w + 2 * (r // 2) - r) // stride + 1
        flops = 6.0 * n * k * p * q * (c // groups) * r * r
        if flops < (3e11 if storage == "f32" else 1.2e12) and max(n * c * h * w, n * k * p * q) < 6e7:
            return {"kind": "conv", "storage": storage, "n": n, "c": c, "h": h, "w": w, "k": k, "r": r, "stride": stride,
                    "pad": r // 2, "groups": groups, "bias": storage == "f32" and rng.random() < 0.5}


def _draw_norm(rng):
    pool, stride, pad, is_max = rng.choice([(3, 2, 1, True), (3, 2, 1, True), (2, 2, 0, True), (2, 2, 0, False)])
    while True:
        n, c, h = _log_int(rng, 2, 128), _log_int(rng, 16, 1024), _log_int(rng, 7, 112)
        w = max(7, min(112, int(h * rng.uniform(0.7, 1.4))))
        if n * c * h * w < 1.1e8:
            return {"kind": "norm", "storage": _chosen(rng, [("f32", 1), ("f16", 1), ("bf16", 1)]), "n": n, "c": c, "h": h, "w": w,
                    "pool": pool, "pool_stride": stride, "pool_pad": pad, "max": is_max}


def _draw_linear(rng):
    while True:
        b, i, o = _log_int(rng, 1, 2048), _log_int(rng, 16, 8192), _log_int(rng, 2, 4096)
        if 6.0 * b * i * o < 6e10:
            return {"kind": "linear", "storage": _chosen(rng, [("f32", 1), ("f16", 1), ("bf16", 1)]), "batch": b, "width": i, "out": o}


def draw(rng):
    return _chosen(rng, [(_draw_train, 8), (_draw_conv, 7), (_draw_norm, 3), (_draw_linear, 2)])(rng)


# ------------------------------------------------------------------------------------ tensors

class _DeviceArray(object):
    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr, "version": 3}


_VIEW_TYPE = {singa.kFloat32: ("<f4", None), singa.kFloat16: ("<f2", None), singa.kBFloat16: ("<i2", torch.bfloat16),
              singa.kInt: ("<i4", None)}


def _torch_view(state, t):
    """The library tensor `t` as a torch tensor over the same memory.  The pool hands memory out again in a short
    cycle, so a state's views are kept by address; what they look at is kept alive by ``state["held"]``."""
    key = (t.ptr, tuple(t.shape()), t.data_type())
    v = state["views"].get(key)
    if v is None:
        typestr, as_type = _VIEW_TYPE[t.data_type()]
        v = torch.as_tensor(_DeviceArray(t.ptr, t.shape(), typestr), device="cuda")
        state["views"][key] = v = v if as_type is None else v.view(as_type)
    return v


def _wrap(dev, t):
    """A torch tensor as a library tensor over the same memory."""
    kind = {torch.float32: singa.kFloat32, torch.float16: singa.kFloat16, torch.bfloat16: singa.kBFloat16,
            torch.int32: singa.kInt}[t.dtype]
    return singa.from_device_pointer(t.data_ptr(), t.shape, dev, kind, keepalive=t)


def _answer(state, **outputs):
    """The outputs of one pass: torch tensors as they are, library tensors through views of their memory."""
    state["held"] = outputs
    return {k: _torch_view(state, v) if isinstance(v, singa.Tensor) else v for k, v in outputs.items()}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, shape, storage="f32", std=1.0):
    return (torch.randn(tuple(shape), generator=gen, device="cuda") * std).to(TORCH_TYPE[storage])


# ------------------------------------------------------------------------------------ networks

class _Draws(object):
    """The random stream the network builders draw their weights from."""

    def __init__(self, seed):
        self.rng = np.random.default_rng(seed)

    def standard_normal(self, shape):
        return self.rng.standard_normal(shape, dtype=np.float32)


class _Arena(object):
    """One flat torch buffer that holds many tensors, each at a 256-byte boundary (a program keeps its parameters
    like this to reduce or save them in one piece)."""

    def __init__(self, dev, tensors, dtype):
        self.dev, self.step = dev, 256 // torch.empty((), dtype=dtype).element_size()
        self.at, total = [], 0
        for t in tensors:
            self.at.append(total)
            total += -(-t.numel() // self.step) * self.step
        self.flat = torch.zeros(max(total, 1), dtype=dtype, device="cuda")
        self.tensors = [self.flat[a:a + t.numel()].view(t.shape).copy_(t) for a, t in zip(self.at, tensors)]

    def wrapped(self):
        return [_wrap(self.dev, t) for t in self.tensors]


def _build(case, ops, seed):
    stream = _Draws(seed)
    if case["net"] == "mlp":
        return workloads.build_mlp(ops, stream, lr=LR, momentum=MOMENTUM, in_dim=case["width"], hidden=case["hidden"],
                                   classes=case["classes"])
    if case["net"] == "cnn":
        return workloads.build_cnn(ops, stream, lr=LR, momentum=MOMENTUM, image=case["image"], c1=case["c1"], c2=case["c2"],
                                   classes=case["classes"])
    build = workloads.build_resnet18 if case["net"] == "resnet18" else workloads.build_resnet50
    return build(ops, stream, lr=LR, momentum=MOMENTUM, classes=case["classes"], final_pool=case["image"] // 32)


def _input_shape(case):
    if case["net"] == "mlp":
        return (case["batch"], case["width"])
    return (case["batch"], 3, case["image"], case["image"])


def _prepare_train(case, seed, dev):
    storage = case["storage"]
    ops = workloads.HipOps(dev) if storage == "f32" else workloads.HalfHipOps(dev, SINGA_TYPE[storage])
    fused = case["tape"] == "fused"
    ops.set_fusion(fused)
    net = _build(case, ops, seed)
    net.sgd.op_by_op = not fused
    gen = _generator(seed)
    x = _wrap(dev, _normal(gen, _input_shape(case), storage))
    labels = _wrap(dev, torch.randint(0, case["classes"], (case["batch"],), generator=gen, device="cuda", dtype=torch.int32))
    # parameters, their fp32 masters and momenta, and the running statistics in flat buffers
    dev.Sync()
    state = {"kind": "train", "views": {}, "net": net, "x": x, "labels": labels, "fused": fused, "forward": case["mode"] == "step"}
    where = [(l, k, l.name + "." + k) for l in net.leaf_layers() for k in l.params]
    values = [_torch_view(state, getattr(l, k)) for l, k, _ in where]
    for l in net.layers:
        if hasattr(l, "sublayers"):   # residual branches start small, as deep networks are trained
            _torch_view(state, (l.bn3 if isinstance(l, workloads.Bottleneck) else l.bn2).scale).fill_(0.2)
    master = _Arena(dev, [v.float() for v in values], torch.float32)
    moment = _Arena(dev, [torch.zeros_like(v, dtype=torch.float32) for v in values], torch.float32)
    short = [i for i, v in enumerate(values) if v.dtype != torch.float32]
    stored = _Arena(dev, [values[i] for i in short], TORCH_TYPE[storage])
    stored_tensors = dict(zip(short, stored.wrapped()))
    for i, ((l, k, name), full, v) in enumerate(zip(where, master.wrapped(), moment.wrapped())):
        net.sgd.moments[name] = v
        if i in stored_tensors:
            net.sgd.masters[name] = full
        setattr(l, k, stored_tensors.get(i, full))
    norms = [l for l in net.leaf_layers() if isinstance(l, workloads.BatchNorm)]
    held = [(l, k) for l in norms for k in ("running_mean", "running_var")]
    running = _Arena(dev, [_torch_view(state, getattr(l, k)) for l, k in held], torch.float32)
    for (l, k), t in zip(held, running.wrapped()):
        setattr(l, k, t)
    # A ReLU gate is a step: a relative change d of its input turns the share d of the gates and moves the gradients behind
    # it by sqrt(d).  Over the 49 ReLUs of a 16-bit ResNet-50, summing a batch in another order alone moves its gradients
    # by 6 to 16 per cent, so there the updated parameters stand for them; momenta are the gradient after one step.
    state["buffers"] = {"parameters": master.flat}
    state["buffers"].update({"stored_parameters": stored.flat} if short else {"momenta": moment.flat})
    state["deep"] = bool(norms)
    if norms:
        state["buffers"]["running_statistics"] = running.flat
    torch.cuda.synchronize()
    state["views"].clear()
    if not state["forward"]:
        net.forward(x, labels)   # the activations that the backward pass finds resident
        dev.Sync()
    return state


def _run_train(state):
    net, out = state["net"], {}
    if state["forward"]:
        out["loss"] = net.forward(state["x"], state["labels"])
    input_gradient = net.backward_and_update(fused_update=state["fused"])
    if not state["deep"]:   # (behind 17 ReLUs single pixels of it move by their own size)
        out["input_gradient"] = input_gradient
    return _answer(state, **dict(out, **state["buffers"]))


def _layers(case):
    """(multiply-adds of one pass, values of the layer's output, weights) of every convolution and dense layer."""
    n, out = case["batch"], []
    if case["net"] == "mlp":
        dims = (case["width"], case["hidden"], case["classes"])
        return [(float(n) * a * b, n * b, a * b + b) for a, b in zip(dims, dims[1:])]

    def conv(c, k, r, size):
        out.append((float(n) * k * size * size * c * r * r, n * k * size * size, c * k * r * r + 2 * k))

    size = case["image"]
    if case["net"] == "cnn":
        conv(3, case["c1"], 5, size)
        conv(case["c1"], case["c2"], 5, size // 2)
        features = case["c2"] * (size // 4) ** 2
    else:
        conv(3, 64, 7, size // 2)
        size, channels = size // 4, 64
        widths, expand = (64, 128, 256, 512), 1 if case["net"] == "resnet18" else 4
        for i, (width, blocks) in enumerate(zip(widths, (2, 2, 2, 2) if expand == 1 else (3, 4, 6, 3))):
            for b in range(blocks):
                step = 2 if i > 0 and b == 0 else 1
                if expand == 1:
                    conv(channels, width, 3, size // step)
                    conv(width, width, 3, size // step)
                else:
                    conv(channels, width, 1, size)
                    conv(width, width, 3, size // step)
                    conv(width, 4 * width, 1, size // step)
                size //= step
                if b == 0 and (step != 1 or channels != width * expand):
                    conv(channels, width * expand, 1, size)
                channels = width * expand
        features = channels
    out.append((float(n) * features * case["classes"], n * case["classes"], (features + 1) * case["classes"]))
    return out


def _work_train(case):
    layers, s = _layers(case), SIZE[case["storage"]]
    step = case["mode"] == "step"
    values, weights = sum(l[1] for l in layers), sum(l[2] for l in layers)
    inputs = int(np.prod(_input_shape(case)))
    # every layer output is stored once by the forward pass and read once by the backward pass; the input is read and its
    # gradient written; parameters and momenta are read and written (16-bit weights beside their masters)
    data = 2 * inputs * s + values * s * (2 if step else 1) + weights * (16 + (4 if s == 2 else 0))
    return {"bytes": float(data), "flops": 2.0 * (3 if step else 2) * sum(l[0] for l in layers)}


# ------------------------------------------------------------------------------------ single layers

def _prepare_conv(case, seed, dev):
    gen, s = _generator(seed), case["storage"]
    c, k, r, groups = case["c"], case["k"], case["r"], case["groups"]
    x = _wrap(dev, _normal(gen, (case["n"], c, case["h"], case["w"]), s))
    W = _wrap(dev, _normal(gen, (k, c // groups, r, r), s, (2.0 / (c // groups * r * r)) ** 0.5))
    b = _wrap(dev, _normal(gen, (k,), s, 0.1)) if case["bias"] else None
    handle = singa.CudnnConvHandle(x, (r, r), (case["stride"],) * 2, (case["pad"],) * 2, c, k, case["bias"], groups)
    dy = _wrap(dev, _normal(gen, (case["n"], k, handle.conv_height, handle.conv_width), s))
    return {"kind": "conv", "views": {}, "x": x, "W": W, "b": b, "dy": dy, "handle": handle}


def _run_conv(state):
    x, W, b, dy, h = (state[k] for k in ("x", "W", "b", "dy", "handle"))
    out = {"y": singa.GpuConvForward(x, W, b, h), "dx": singa.GpuConvBackwardx(dy, W, x, h),
           "dW": singa.GpuConvBackwardW(dy, x, W, h)}
    if b is not None:
        out["db"] = singa.GpuConvBackwardb(dy, b, h)
    return _answer(state, **out)


def _work_conv(case):
    r, st, pad = case["r"], case["stride"], case["pad"]
    p, q = (case["h"] + 2 * pad - r) // st + 1, (case["w"] + 2 * pad - r) // st + 1
    x, y = case["n"] * case["c"] * case["h"] * case["w"], case["n"] * case["k"] * p * q
    w = case["k"] * (case["c"] // case["groups"]) * r * r
    return {"bytes": float(2 * (x + y + w) * SIZE[case["storage"]]), "flops": 6.0 * y * (case["c"] // case["groups"]) * r * r}


def _prepare_norm(case, seed, dev):
    gen, s = _generator(seed), case["storage"]
    shape, c = (case["n"], case["c"], case["h"], case["w"]), case["c"]
    x = _wrap(dev, (torch.randn(shape, generator=gen, device="cuda") * 1.5 + 0.3).to(TORCH_TYPE[s]))
    scale, bias = _wrap(dev, 1 + _normal(gen, (c,), std=0.2)), _wrap(dev, _normal(gen, (c,), std=0.2))
    running = [torch.zeros(c, device="cuda"), torch.ones(c, device="cuda")]
    norm = singa.CudnnBatchNormHandle(0.9, x)
    pool = singa.CudnnPoolingHandle(x, (case["pool"],) * 2, (case["pool_stride"],) * 2, (case["pool_pad"],) * 2, case["max"])
    state = {"kind": "norm", "views": {}, "x": x, "scale": scale, "bias": bias, "running": running, "norm": norm, "pool": pool,
             "wrapped": [_wrap(dev, t) for t in running], "dy": _wrap(dev, _normal(gen, shape, s))}
    # the pooling layer's input: an activation behind a ReLU (half of it zeros, hence ties)
    state["a"] = _wrap(dev, _normal(gen, shape, s).clamp_(min=0))
    state["dz"] = _wrap(dev, _normal(gen, (case["n"], c, pool.pooled_height, pool.pooled_width), s))
    return state


def _run_norm(state):
    x, scale, bias, norm, pool = (state[k] for k in ("x", "scale", "bias", "norm", "pool"))
    mean, var = state["wrapped"]
    y, saved_mean, saved_var = singa.GpuBatchNormReLUForwardTraining(norm, x, scale, bias, mean, var)
    z = singa.GpuPoolingForward(pool, state["a"])
    da = singa.GpuPoolingBackward(pool, state["dz"], state["a"], z)
    dx, dscale, dbias = singa.GpuBatchNormReLUBackward(norm, state["dy"], x, scale, bias, saved_mean, saved_var)
    return _answer(state, y=y, z=z, da=da, dx=dx, dscale=dscale, dbias=dbias, mean=saved_mean, inverse_std=saved_var,
                   running_mean=state["running"][0], running_var=state["running"][1])


def _work_norm(case):
    x = case["n"] * case["c"] * case["h"] * case["w"]
    z = x // case["pool_stride"] ** 2
    # forward: x in, y out; a in, z out; backward: dz and a in, da out; dy and x in, dx out
    return {"bytes": float((8 * x + 2 * z) * SIZE[case["storage"]]), "flops": 20.0 * x}


def _prepare_linear(case, seed, dev):
    gen, s = _generator(seed), case["storage"]
    b, i, o = case["batch"], case["width"], case["out"]
    state = {"kind": "linear", "views": {}, "x": _wrap(dev, _normal(gen, (b, i), s)),
             "W": _wrap(dev, _normal(gen, (i, o), s, (2.0 / i) ** 0.5)), "dy": _wrap(dev, _normal(gen, (b, o), s)), "b": None}
    if s == "f32":   # (the row functions of the bias are fp32 functions)
        state["b"] = _wrap(dev, _normal(gen, (o,), s, 0.1))
    return state


def _run_linear(state):
    x, W, b, dy = (state[k] for k in ("x", "W", "b", "dy"))
    out = {"y": singa.Mult(x, W)}
    if b is not None:
        singa.AddRow(b, out["y"])
        out["db"] = singa.Sum(dy, 0)
    out["dx"] = singa.Mult(dy, singa.DefaultTranspose(W))
    out["dW"] = singa.Mult(singa.DefaultTranspose(x), dy)
    return _answer(state, **out)


def _work_linear(case):
    b, i, o = case["batch"], case["width"], case["out"]
    return {"bytes": float(2 * (b * i + i * o + b * o) * SIZE[case["storage"]]), "flops": 6.0 * b * i * o}


# ------------------------------------------------------------------------------------ the five functions

_PREPARE = {"train": _prepare_train, "conv": _prepare_conv, "norm": _prepare_norm, "linear": _prepare_linear}
_RUN = {"train": _run_train, "conv": _run_conv, "norm": _run_norm, "linear": _run_linear}
_WORK = {"train": _work_train, "conv": _work_conv, "norm": _work_norm, "linear": _work_linear}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed, singa.create_hip_gpu_on(0))
    torch.cuda.synchronize()   # the library works on streams of its own: what torch has made is there before they start
    return state


def run(state):
    return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


# About four times what another order of the sums shows.  Networks: the images of a batch permuted and, in fp32, the weights
# moved by 1e-7 of themselves, after two passes; the values are those of the gates that turn (see _prepare_train) in fp32, and
# of the loss and the running statistics in 16 bits.  Layers: against float64; in 16 bits one rounding of the result.
_TOLERANCE = {
    "mlp": {"rel": 1e-3, "max": 0.2},
    "cnn": {"rel": 8e-3, "max": 0.99},
    "resnet18": {"rel": 1e-2, "max": 0.99},
    "resnet50 f16": {"rel": 2e-3, "max": 1.6e-2},
    "resnet50 bf16": {"rel": 8e-3, "max": 6e-2},
    "layer f32": {"rel": 6e-6, "max": 4e-5},
    "layer f16": {"rel": 8e-4, "max": 4e-3},
    "layer bf16": {"rel": 7e-3, "max": 3e-2},
}


def tolerance(case):
    name = case["net"] if case["kind"] == "train" else "layer"
    return dict(_TOLERANCE[name if name in _TOLERANCE else name + " " + case["storage"]])
