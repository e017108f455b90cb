"""Timing cases of the training engine: single layers, blocks, optimiser steps
and whole training steps, each through the public nn_engine API.

listed() names the cases, draw(rng) gives more of the same ranges, prepare()
builds what a program holds before the call, run() is one pass, work() the
bytes and operations the pass cannot do without, tolerance() how far two
correct fp32 implementations may differ, exact() the same outputs in 64 bits
from plain torch.

Gradients behind a ReLU, ReLU6 or max-pool have no 64-bit value to compare
with: an activation within fp32 rounding of the decision sends its whole
gradient the one way or the other, whichever implementation rounds it.  A
handful of such elements in a layer of 10^7 moves the layer's gradients by
1e-4 to 1e-3 (2-norm).  exact() gives None for those outputs, and the
tolerance of those cases covers a few flipped decisions; the cases without an
activation pin the products themselves.
"""
import ctypes
import math

import torch
import torch.nn.functional as F

from directcompute_torch_amd import nn_engine as nn

GPU = "cuda"


# --------------------------------------------------------------------------
# Device memory: a buffer handle is a pointer to a record whose first field is
# the device pointer (include/dcengine.h), so torch can fill and read the
# engine's buffers in place.
# --------------------------------------------------------------------------
class _Span:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False),
                                         "strides": None, "version": 2}


def _view(t):
    """The engine tensor's device memory as a torch tensor (no copy)."""
    ptr = ctypes.cast(t.gpu_buf, ctypes.POINTER(ctypes.c_void_p))[0]
    return torch.as_tensor(_Span(ptr, t.shape), device=GPU)


def _to_engine(a, grad=False):
    t = nn.Tensor.empty(tuple(a.shape), requires_grad=grad, track=False)
    _view(t).copy_(a)
    return t


# --------------------------------------------------------------------------
# Networks, written once over a small op interface: `Engine` runs nn_engine,
# `Exact` plain torch in float64.
# --------------------------------------------------------------------------
class Engine:
    def __init__(self, params):
        self.P = {k: _to_engine(v, grad=True) for k, v in params.items()}
        self.stats = {}

    def conv(self, x, name, s=1, p=0, act=0):
        return nn.conv2d(x, self.P[name + ".w"], self.P[name + ".b"], s, p, act)

    def depthwise(self, x, name, s, p):
        return nn.depthwise_conv2d(x, self.P[name + ".w"], self.P[name + ".b"], s, p)

    def linear(self, x, name, relu):
        m = nn.matmul(x, self.P[name + ".w"])
        return nn.bias_relu(m, self.P[name + ".b"]) if relu else nn.add_bias(m, self.P[name + ".b"])

    def bn(self, x, name):
        if name not in self.stats:
            c = x.shape[1]
            self.stats[name] = (nn.Tensor([0.0] * c, track=False), nn.Tensor([1.0] * c, track=False))
        return nn.batchnorm2d(x, self.P[name + ".g"], self.P[name + ".be"], *self.stats[name])

    relu, relu6, sigmoid = staticmethod(nn.relu), staticmethod(nn.relu6), staticmethod(nn.sigmoid)
    maxpool, upsample, flatten = staticmethod(nn.maxpool2d), staticmethod(nn.upsample2d), staticmethod(nn.flatten)
    add, concat = staticmethod(nn.add), staticmethod(nn.concat)
    cross_entropy, dice = staticmethod(nn.softmax_ce), staticmethod(nn.dice_loss)


class Exact:
    def __init__(self, params):
        self.P = {k: v.double().requires_grad_(True) for k, v in params.items()}

    def conv(self, x, name, s=1, p=0, act=0, groups=1):
        y = F.conv2d(x, self.P[name + ".w"], self.P[name + ".b"], stride=s, padding=p, groups=groups)
        return F.relu(y) if act else y

    def depthwise(self, x, name, s, p):
        return self.conv(x, name, s, p, groups=x.shape[1])

    def linear(self, x, name, relu):
        y = x @ self.P[name + ".w"] + self.P[name + ".b"]
        return F.relu(y) if relu else y

    def bn(self, x, name):
        mean, var = x.mean((0, 2, 3), keepdim=True), x.var((0, 2, 3), unbiased=False, keepdim=True)
        g, be = (self.P[name + k].view(1, -1, 1, 1) for k in (".g", ".be"))
        return (x - mean) / torch.sqrt(var + 1e-5) * g + be

    relu, sigmoid = staticmethod(F.relu), staticmethod(torch.sigmoid)
    relu6, maxpool = staticmethod(F.relu6), staticmethod(F.max_pool2d)

    def upsample(self, x):
        return x.repeat_interleave(2, 2).repeat_interleave(2, 3)

    def flatten(self, x):
        return x.flatten(1)

    def add(self, a, b):
        return a + b

    def concat(self, ts):
        return torch.cat(ts, 1)

    def cross_entropy(self, z, labels):
        return F.cross_entropy(z, labels.long()).reshape(1)

    def dice(self, p, t):
        p, t = p.flatten(1), t.flatten(1)
        return 1 - 2 * (p * t).sum(1) / (p.sum(1) + t.sum(1) + 1e-6)


def _conv_p(out, name, cin, cout, k, depthwise=False):
    out[name + ".w"] = ((cout, 1 if depthwise else cin, k, k), math.sqrt(2.0 / ((1 if depthwise else cin) * k * k)), 0.0)
    out[name + ".b"] = ((cout,), 0.01, 0.0)


def _bn_p(out, name, c):
    out[name + ".g"] = ((c,), 0.1, 1.0)
    out[name + ".be"] = ((c,), 0.1, 0.0)


def _linear_p(out, name, fin, fout):
    out[name + ".w"] = ((fin, fout), math.sqrt(2.0 / fin), 0.0)
    out[name + ".b"] = ((fout,), 0.01, 0.0)


LENET = [("c1", 1, 6), ("c2", 6, 16)]
LENET_FC = [("l1", 256, 120), ("l2", 120, 84), ("l3", 84, 10)]
ALEXNET = [("c1", 3, 64, 11, 4, 2), ("c2", 64, 192, 5, 1, 2), ("c3", 192, 384, 3, 1, 1),
           ("c4", 384, 256, 3, 1, 1), ("c5", 256, 256, 3, 1, 1)]
ALEXNET_FC = [("l1", 9216, 4096), ("l2", 4096, 4096), ("l3", 4096, 1000)]
UNET_BASE, UNET_LEVELS = 16, 4


def _unet_convs():
    """(name, in, out, halvings of the image) of UNet-base16's 3x3 layers."""
    got, prev = [], 3
    for i in range(UNET_LEVELS):
        c = UNET_BASE << i
        got += [("e%da" % i, prev, c, i), ("e%db" % i, c, c, i)]
        prev = c
    c = UNET_BASE << UNET_LEVELS
    got += [("ba", prev, c, UNET_LEVELS), ("bb", c, c, UNET_LEVELS)]
    prev = c
    for i in reversed(range(UNET_LEVELS)):
        c = UNET_BASE << i
        got += [("d%da" % i, prev + c, c, i), ("d%db" % i, c, c, i)]
        prev = c
    return got


def _param_specs(case):
    """{name: (shape, spread, centre)} of the case's parameters."""
    p, kind = {}, case["kind"]
    if kind == "conv":
        _conv_p(p, "c", case["cin"], case["cout"], case["k"])
    elif kind == "linear":
        _linear_p(p, "l", case["fin"], case["fout"])
    elif kind == "block":
        h = 6 * case["cin"]
        _conv_p(p, "exp", case["cin"], h, 1)
        _bn_p(p, "bn1", h)
        _conv_p(p, "dw", h, h, 3, depthwise=True)
        _bn_p(p, "bn2", h)
        _conv_p(p, "proj", h, case["cout"], 1)
        _bn_p(p, "bn3", case["cout"])
    elif kind == "update":
        for i, n in enumerate(_split(case["values"], case["tensors"])):
            p["w%d" % i] = ((n,), 0.02, 0.0)
    elif case["model"] == "lenet":
        for n, ci, co in LENET:
            _conv_p(p, n, ci, co, 5)
        for n, fi, fo in LENET_FC:
            _linear_p(p, n, fi, fo)
    elif case["model"] == "alexnet":
        for n, ci, co, k, _, _ in ALEXNET:
            _conv_p(p, n, ci, co, k)
        for n, fi, fo in ALEXNET_FC:
            _linear_p(p, n, fi, fo)
    else:
        for n, ci, co, _ in _unet_convs():
            _conv_p(p, n, ci, co, 3)
            _bn_p(p, n + ".bn", co)
        _conv_p(p, "head", UNET_BASE, 1, 1)
    return p


def _split(values, tensors):
    """Tensor sizes as networks have them: each about half of the one before
    (a big matrix, smaller ones, and biases of a few values), none empty."""
    got, left = [], values
    for i in range(tensors - 1):
        n = max(1, min(left - (tensors - 1 - i), left * 5 // 9))
        got.append(n)
        left -= n
    return got + [left]


def _lenet(net, x):
    for n, _, _ in LENET:
        x = net.maxpool(net.conv(x, n, act=1), 2, 2)
    x = net.flatten(x)
    for n, _, fo in LENET_FC:
        x = net.linear(x, n, fo != 10)
    return x


def _alexnet(net, x):
    for n, _, _, _, s, p in ALEXNET:
        x = net.conv(x, n, s, p, 1)
        if n in ("c1", "c2", "c5"):
            x = net.maxpool(x, 3, 2)
    x = net.flatten(x)
    for n, _, fo in ALEXNET_FC:
        x = net.linear(x, n, fo != 1000)
    return x


def _unet(net, x):
    def cbr(h, name):
        return net.relu(net.bn(net.conv(h, name, 1, 1), name + ".bn"))
    skips = []
    for i in range(UNET_LEVELS):
        x = cbr(cbr(x, "e%da" % i), "e%db" % i)
        skips.append(x)
        x = net.maxpool(x, 2, 2)
    x = cbr(cbr(x, "ba"), "bb")
    for i in reversed(range(UNET_LEVELS)):
        x = cbr(cbr(net.concat([net.upsample(x), skips[i]]), "d%da" % i), "d%db" % i)
    return net.sigmoid(net.conv(x, "head"))


NETS = {"lenet": _lenet, "alexnet": _alexnet, "unet": _unet}


def _layer(net, case, x):
    """The output of a layer or block case."""
    if case["kind"] == "conv":
        return net.conv(x, "c", case["stride"], case["pad"], case["relu"])
    if case["kind"] == "linear":
        return net.linear(x, "l", bool(case["relu"]))
    t = net.relu6(net.bn(net.conv(x, "exp"), "bn1"))
    t = net.relu6(net.bn(net.depthwise(t, "dw", case["stride"], 1), "bn2"))
    t = net.bn(net.conv(t, "proj"), "bn3")
    return net.add(t, x) if case["stride"] == 1 and case["cin"] == case["cout"] else t


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
def _conv(batch, cin, h, w, cout, k, stride, pad, relu, first=0):
    return dict(kind="conv", batch=batch, cin=cin, h=h, w=w, cout=cout, k=k, stride=stride, pad=pad, relu=relu, first=first)


def _block(batch, cin, cout, h, w, stride):
    return dict(kind="block", batch=batch, cin=cin, cout=cout, h=h, w=w, stride=stride)


def _linear(rows, fin, fout, relu):
    return dict(kind="linear", rows=rows, fin=fin, fout=fout, relu=relu)


def _update(rule, values, tensors, norm):
    return dict(kind="update", rule=rule, values=values, tensors=tensors, norm=norm)


def _step(model, batch, size, replay=0):
    return dict(kind="step", model=model, batch=batch, size=size, replay=replay)


def listed():
    return [
        # The smallest training step: LeNet-5, SGD, dispatched call by call.  Launches and host calls.
        dict(_step("lenet", 64, 28), name="lenet_step_b64"),
        # The same step recorded once with ComputeGraph and replayed: launches alone.
        dict(_step("lenet", 64, 28, replay=1), name="lenet_replay_b64"),
        # The flagship: a whole AlexNet-224 step with AdamW at batch 128.
        dict(_step("alexnet", 128, 224), name="alexnet_step_b128"),
        # Segmentation: UNet-base16 at 256x256 with batch norm, Dice loss, global norm clip and Adam.
        dict(_step("unet", 8, 256), name="unet_step_b8"),
        # The 3x3 layer over a large image (VGG and ResNet stems), forward and backward.
        dict(_conv(128, 64, 56, 56, 128, 3, 1, 1, 0), name="conv3_64_128_56"),
        # A network's first layer: 11x11 stride 4 over RGB with ReLU; no input gradient.
        dict(_conv(128, 3, 224, 224, 64, 11, 4, 2, 1, first=1), name="conv11_3_64_224_relu"),
        # The deep 3x3 layer over a small odd image with ReLU.
        dict(_conv(128, 192, 13, 13, 384, 3, 1, 1, 1), name="conv3_192_384_13_relu"),
        # A pointwise expansion, as inverted residual blocks have them.
        dict(_conv(64, 24, 56, 56, 144, 1, 1, 0, 0), name="conv1_24_144_56"),
        # Odd everything: a ragged image, channels that fill no tile, 5x5 at stride 2.
        dict(_conv(12, 37, 61, 45, 70, 5, 2, 2, 0), name="conv5s2_37_70_ragged"),
        # The largest fully connected layer of AlexNet, forward and backward.
        dict(_linear(128, 9216, 4096, 1), name="linear_9216_4096"),
        # One inverted residual block at 112x112: pointwise, batch norm, ReLU6, depthwise, forward and backward.
        dict(_block(64, 16, 24, 112, 112, 2), name="block_16_24_112"),
        # The parameter update of a 62 M parameter network after its gradients, with their norm.
        dict(_update("adamw", 62378344, 16, 1), name="adamw_62m_norm"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "conv", "linear", "linear", "block", "block", "update", "step", "step"])
    if kind == "conv":
        while True:
            k = rng.choice([1, 3, 3, 3, 5])
            first = int(rng.random() < 0.15)
            c = dict(_conv(_log(rng, 1, 128), 3 if first else _log(rng, 8, 384), _log(rng, 7, 160), _log(rng, 7, 160),
                           _log(rng, 8, 384), k, rng.choice([1, 1, 1, 2]), rng.choice([0, k // 2, k // 2]),
                           rng.choice([0, 1]), first))
            w = work(c)
            if 2e8 < w["flops"] < 2.5e11 and w["bytes"] < 2e9:
                return c
    if kind == "linear":
        return _linear(_log(rng, 1, 512), _log(rng, 64, 9216), _log(rng, 10, 4096), rng.choice([0, 1]))
    if kind == "block":
        ci = rng.choice([8, 16, 20, 24, 32])
        return _block(_log(rng, 1, 64), ci, rng.choice([ci, 24, 32, 40]), _log(rng, 14, 112), _log(rng, 14, 112), rng.choice([1, 2]))
    if kind == "update":
        return _update(rng.choice(["adamw", "sgd"]), _log(rng, 40000, 62378344), rng.randint(4, 20), rng.choice([0, 1]))
    model = rng.choice(["lenet", "alexnet", "unet"])
    if model == "lenet":
        return _step("lenet", _log(rng, 1, 512), 28, rng.choice([0, 1]))
    if model == "alexnet":
        return _step("alexnet", _log(rng, 4, 127), 224)
    return _step("unet", rng.randint(1, 8), 16 * rng.randint(4, 15))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _out_hw(c):
    k, s, p = (c["k"], c["stride"], c["pad"]) if c["kind"] == "conv" else (3, c["stride"], 1)
    return (c["h"] + 2 * p - k) // s + 1, (c["w"] + 2 * p - k) // s + 1


def _data(case, seed):
    """The case's inputs as torch tensors on the GPU: params, and x, dy or labels."""
    g = torch.Generator(device=GPU)
    g.manual_seed(seed)

    def normal(shape, spread=1.0, centre=0.0):
        return torch.randn(shape, generator=g, device=GPU).mul_(spread).add_(centre)

    d = {"params": {k: normal(*v) for k, v in _param_specs(case).items()}}
    kind = case["kind"]
    if kind == "update":
        # gradients of a norm near 1, as they come from a backward pass
        d["grads"] = [normal(v.shape, 1 / math.sqrt(case["values"])) for v in d["params"].values()]
        # a running optimiser: second moments of gradients of this size
        d["m"] = [normal(v.shape, 0.3 / math.sqrt(case["values"])) for v in d["params"].values()]
        d["v"] = [normal(v.shape).square_().mul_(0.5 / case["values"]) for v in d["params"].values()]
    elif kind == "linear":
        d["x"] = normal((case["rows"], case["fin"])).clamp_(min=0.0)  # a ReLU's output
        d["dy"] = normal((case["rows"], case["fout"]), 1 / case["rows"])
    elif kind in ("conv", "block"):
        d["x"] = normal((case["batch"], case["cin"], case["h"], case["w"]))
        if kind == "conv" and not case["first"]:
            d["x"].clamp_(min=0.0)
        d["dy"] = normal((case["batch"], case["cout"]) + _out_hw(case), 1 / case["batch"])
    elif case["model"] == "unet":
        n = case["size"]
        d["x"] = torch.rand((case["batch"], 3, n, n), generator=g, device=GPU)
        blobs = (torch.rand((case["batch"], 1, n // 8, n // 8), generator=g, device=GPU) < 0.3).float()
        d["labels"] = blobs.repeat_interleave(8, 2).repeat_interleave(8, 3)
    else:
        d["x"] = normal((case["batch"], 1 if case["model"] == "lenet" else 3, case["size"], case["size"]))
        top = 10 if case["model"] == "lenet" else 1000
        d["labels"] = torch.randint(0, top, (case["batch"],), generator=g, device=GPU).float()
    return d


def _optimizer(case, params):
    if case["kind"] == "update":
        return nn.SGD(params, lr=0.01) if case["rule"] == "sgd" else nn.AdamW(params, lr=1e-4, weight_decay=0.01)
    if case["model"] == "lenet":
        return nn.SGD(params, lr=0.01)
    if case["model"] == "alexnet":
        return nn.AdamW(params, lr=1e-4, weight_decay=0.01)
    return nn.Adam(params, lr=1e-3)


def prepare(case, seed):
    d = _data(case, seed)
    net = Engine(d["params"])
    s = {"case": case, "net": net, "params": list(net.P.values())}
    kind = case["kind"]
    if kind in ("conv", "linear", "block"):
        s["x"] = _to_engine(d["x"], grad=not case.get("first"))
        s["dy"] = _to_engine(d["dy"])
    elif kind == "update":
        s["grads"] = [_to_engine(g) for g in d["grads"]]
        s["opt"] = opt = _optimizer(case, s["params"])
        if case["rule"] == "adamw":
            opt.t = 100
            for have, want in zip(opt.m + opt.v, d["m"] + d["v"]):
                _view(have).copy_(want)
    else:
        s["opt"] = _optimizer(case, s["params"])
        if case["replay"]:
            s["graph"] = nn.ComputeGraph()
            before = {k: _to_engine(v) for k, v in d["params"].items()}

            def forward(x):  # keeps a reference of its own on the logits of the recorded step
                out = NETS[case["model"]](net, x)
                nn.lib.AddRefBuffer(out.gpu_buf)
                s["logits"] = nn.Tensor.from_gpu(out.gpu_buf, out.shape, track=False)
                return out
            s["graph"].trace(forward, s["opt"], d["x"].cpu().numpy(), d["labels"].cpu().numpy(), s["params"], clip=1.0)
            nn.sync_gpu()
            for k, t in net.P.items():  # tracing trains one batch: start from the weights as given
                _view(t).copy_(_view(before[k]))
        else:
            s["x"], s["labels"] = _to_engine(d["x"]), _to_engine(d["labels"])
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
# The bias of a convolution that a batch norm follows has a gradient of zero;
# what comes out is the rounding of its sum, which no two implementations
# share.  It is computed, and not compared.
def _compared(case, names):
    if case["kind"] == "block":
        return [n for n in names if n not in ("exp.b", "dw.b", "proj.b")]
    if case["kind"] == "step" and case["model"] == "unet":
        return [n for n in names if not n.endswith(".b") or n == "head.b"]
    return list(names)


def run(s):
    case, net = s["case"], s["net"]
    kind = case["kind"]
    if kind == "step" and case["replay"]:
        s["graph"].replay()
        return {"logits": _view(s["logits"]), "params": [_view(t) for t in s["params"]]}
    nn.end_batch()  # the previous batch's buffers, as a training loop does after each batch
    for t in s["params"]:
        t.grad = None
    names = _compared(case, net.P)
    if kind in ("conv", "linear", "block"):
        s["x"].grad = None
        y = _layer(net, case, s["x"])
        y.backward(s["dy"])
        out = {"y": _view(y), "grads": [_view(net.P[n].grad) for n in names]}
        if not case.get("first"):
            out["dx"] = _view(s["x"].grad)
        return out
    opt = s["opt"]
    if kind == "update":
        for t, g in zip(s["params"], s["grads"]):
            t.grad = g
        out = {"params": [_view(t) for t in s["params"]]}
        if case["norm"]:
            out["norm"] = nn.clip_grad_norm(s["params"], 2.0)
        opt.step(clip=1.0)
        if case["rule"] == "adamw":
            out["m"], out["v"] = [_view(t) for t in opt.m], [_view(t) for t in opt.v]
        return out
    out = NETS[case["model"]](net, s["x"])
    loss = (net.dice if case["model"] == "unet" else net.cross_entropy)(out, s["labels"])
    loss.backward()
    if case["model"] == "unet":
        nn.clip_grad_norm(s["params"], 1.0)
    opt.step(clip=1.0)
    got = {"logits": _view(out), "loss": _view(loss), "grads": [_view(net.P[n].grad) for n in names]}
    if case["model"] != "unet":
        got["params"] = [_view(t) for t in s["params"]]
    return got


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def _prod(shape):
    n = 1
    for d in shape:
        n *= d
    return n


def work(case):
    kind = case["kind"]
    n_params = sum(_prod(v[0]) for v in _param_specs(case).values())
    if kind == "conv":
        oh, ow = _out_hw(case)
        x, y = case["batch"] * case["cin"] * case["h"] * case["w"], case["batch"] * case["cout"] * oh * ow
        # in: x, w, b, dy; out: y, dw, db, dx
        products = 2 if case["first"] else 3
        return {"bytes": 4.0 * ((products - 1) * x + 2 * y + 2 * n_params),
                "flops": 2.0 * products * y * case["cin"] * case["k"] ** 2}
    if kind == "linear":
        r, fi, fo = case["rows"], case["fin"], case["fout"]
        return {"bytes": 4.0 * (2 * r * fi + 2 * r * fo + 2 * n_params), "flops": 6.0 * r * fi * fo}
    if kind == "block":
        oh, ow = _out_hw(case)
        big, small = case["h"] * case["w"], oh * ow
        hid = 6 * case["cin"]
        # x, dy in; y, dx out; the three normalised tensors are kept from the forward for the backward
        values = case["batch"] * (2 * case["cin"] * big + 2 * case["cout"] * small
                                  + 2 * (hid * big + hid * small + case["cout"] * small))
        flops = 6.0 * case["batch"] * hid * (case["cin"] * big + 9 * small + case["cout"] * small)
        return {"bytes": 4.0 * (values + 2 * n_params), "flops": flops}
    if kind == "update":
        return {"bytes": (28.0 if case["rule"] == "adamw" else 12.0) * n_params, "flops": 12.0 * n_params}
    b, layers = case["batch"], []  # (values of a layer's output, products per value, gradient of the input too)
    if case["model"] == "lenet":
        layers += [(6 * 24 * 24, 25, 0), (16 * 8 * 8, 150, 1)] + [(fo, fi, 1) for _, fi, fo in LENET_FC]
        state = 3  # w in, w out, gradient out
    elif case["model"] == "alexnet":
        for (_, ci, co, k, _, _), hw in zip(ALEXNET, (55, 27, 13, 13, 13)):
            layers.append((co * hw * hw, ci * k * k, ci != 3))
        layers += [(fo, fi, 1) for _, fi, fo in ALEXNET_FC]
        state = 7
    else:
        for _, ci, co, i in _unet_convs():
            layers.append((co * (case["size"] >> i) ** 2, 9 * ci, ci != 3))
        layers.append((case["size"] ** 2, UNET_BASE, 1))
        state = 7
    flops = sum(2.0 * b * n * k * (2 + dx) for n, k, dx in layers)
    # each layer's output is written in the forward and read in the backward
    values = 2 * b * sum(n for n, _, _ in layers)
    return {"bytes": 4.0 * (values + state * n_params), "flops": flops}


# --------------------------------------------------------------------------
# How far two correct fp32 implementations may differ
# --------------------------------------------------------------------------
# Four times what the outputs were off by against float64 over two seeds and a
# few drawn cases: sums in fp32 alone (products and updates), or sums and the
# few decisions that their rounding turns (see the top of the file): up to
# 7e-4 in a layer or block, 5.5e-3 in AlexNet's first gradient and 6.7e-3 in a
# batch-normed UNet, where a turned decision also moves the statistics of
# every layer before it.
def tolerance(case):
    if case["kind"] == "step":
        if case["replay"]:
            return {"rel": 4e-5, "max": 1e-3}
        return {"rel": 2.5e-2, "max": 0.95}
    if case["kind"] == "block":
        return {"rel": 3e-3, "max": 0.95}
    if case["kind"] == "update":
        return {"rel": 4e-7, "max": 5e-5}
    if case["relu"]:
        return {"rel": 3e-3, "max": 0.5}
    return {"rel": 3e-6, "max": 4e-5}


def _exact(case, seed):
    """Every output of the first pass in float64."""
    d = _data(case, seed)
    kind = case["kind"]
    if kind == "update":
        return _exact_update(case, d)
    net = Exact(d["params"])
    names = _compared(case, net.P)
    with torch.backends.cudnn.flags(enabled=False):  # float64 convolutions run in torch's own code
        x = d["x"].double().requires_grad_(kind != "step" and not case.get("first"))
        if kind != "step":
            y = _layer(net, case, x)
            y.backward(d["dy"].double())
            out = {"y": y.detach(), "grads": [net.P[n].grad for n in names]}
            if not case.get("first"):
                out["dx"] = x.grad
            return out
        y = NETS[case["model"]](net, x)
        loss = (net.dice if case["model"] == "unet" else net.cross_entropy)(y, d["labels"].double())
        loss.mean().backward()
    grads = [p.grad for p in net.P.values()]
    if case["model"] == "unet":
        norm = math.sqrt(sum(float(g.square().sum()) for g in grads))
        if norm > 1.0:
            for g in grads:
                g.mul_(1.0 / (norm + 1e-6))
        return {"logits": y.detach(), "loss": loss.detach(), "grads": [net.P[n].grad for n in names]}
    out = {"logits": y.detach(), "loss": loss.detach(), "grads": grads}
    zero = [torch.zeros_like(g) for g in grads]
    ps = [p.detach() for p in net.P.values()]
    if case["model"] == "lenet":
        out["params"] = [p - 0.01 * g.clamp(-1, 1) for p, g in zip(ps, grads)]
    else:
        out["params"] = [_adamw(p, g, m, m, 1)[0] for p, g, m in zip(ps, grads, zero)]
    return {k: out[k] for k in ("logits", "params")} if case["replay"] else out


def _adamw(p, g, m, v, t, lr=1e-4, wd=0.01):
    g = g.clamp(-1, 1)
    m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
    size = lr * math.sqrt(1 - 0.999 ** t) / (1 - 0.9 ** t)
    return p - lr * wd * p - size * m / (v.sqrt() + 1e-8), m, v


def _exact_update(case, d):
    ps, gs = [p.double() for p in d["params"].values()], [g.double() for g in d["grads"]]
    out = {}
    if case["norm"]:
        norm = math.sqrt(sum(float(g.square().sum()) for g in gs))
        out["norm"] = norm
        if norm > 2.0:
            gs = [g * (2.0 / (norm + 1e-6)) for g in gs]
    if case["rule"] == "sgd":
        out["params"] = [p - 0.01 * g.clamp(-1, 1) for p, g in zip(ps, gs)]
        return out
    got = [_adamw(p, g, m.double(), v.double(), 101) for p, g, m, v in zip(ps, gs, d["m"], d["v"])]
    out["params"], out["m"], out["v"] = ([r[k] for r in got] for k in range(3))
    return out


def exact(case, seed):
    out = _exact(case, seed)
    if case["kind"] in ("block", "step") or case.get("relu"):  # gradients behind a decision: see above
        return {k: v if k in ("y", "logits", "loss") else None if torch.is_tensor(v) else [None] * len(v) for k, v in out.items()}
    return out
