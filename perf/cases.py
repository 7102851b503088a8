"""What this framework's speed is measured on: calls of its public entry points.

Two groups of entry points are covered:

* the layer (``torch_ops.CP4Conv2d``), as a network uses it: inference under
  ``torch.no_grad()``, or one training step - forward, then backward to the input
  gradient, the four factor gradients and the bias gradient;
* the three passes of the binding (``conv2d_forward``, ``conv2d_backward_data``,
  ``conv2d_backward_filter``), as a program that keeps its own buffers calls them.

Sizes are those of the five workloads in ``paralleltnnlayers_amd.configs``, of the
shape lists under ``csrc/host/shapes`` and of the tests.  ``draw`` covers what lies
between: 1 to 128 images, planes of 7 x 7 to 512 x 512 with odd and unequal sides, 1 to
512 channels, ranks 1 to 64, filters 1, 3, 5 (and 7 without a filter gradient), fp32
and both 16-bit activation types, stride 1 and 2.
"""
import math

import torch

import paralleltnnlayers_amd as cp4
from paralleltnnlayers_amd import torch_ops

# what a case does: the layer's inference and training step, the binding's passes
INFER, STEP = "infer", "step"
FORWARD, BACKWARD_DATA, BACKWARD_FILTER = "forward", "backward_data", "backward_filter"

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _case(name, op, N, C, H, W, T, k, R, dtype="f32", stride=1, first=False):
    return dict(name=name, op=op, N=N, C=C, H=H, W=W, T=T, k=k, R=R, dtype=dtype,
                stride=stride, first=first)


def listed():
    return [
        # one small image through one layer: nothing but latency (workload C1)
        _case("fwd_1x16x32x32_r8", FORWARD, 1, 16, 32, 32, 16, 3, 8),
        # the last layer of AlexNet's list on one image: an odd plane, few pixels, bias
        # and ReLU fused
        _case("infer_1x192x13x13_r16", INFER, 1, 192, 13, 13, 256, 3, 16),
        # a VGG-16 block on a batch of 8 in half precision: wide planes, inference
        _case("infer_8x64x224x224_r16_f16", INFER, 8, 64, 224, 224, 64, 3, 16, dtype="f16"),
        # a middle layer of a small network (workload C2's shape), trained
        _case("step_16x64x32x32_r16", STEP, 16, 64, 32, 32, 64, 3, 16),
        # a ResNet stage's shape (workload C3): the forward pass, then the whole step
        _case("fwd_32x256x56x56_r32", FORWARD, 32, 256, 56, 56, 256, 3, 32),
        _case("step_32x256x56x56_r32", STEP, 32, 256, 56, 56, 256, 3, 32),
        # input gradient under a 5 x 5 filter (workload C4)
        _case("bdata_32x128x28x28_r16", BACKWARD_DATA, 32, 128, 28, 28, 128, 5, 16),
        # factor gradients of small planes at a high rank (workload C5)
        _case("bfilter_64x256x14x14_r64", BACKWARD_FILTER, 64, 256, 14, 14, 256, 3, 64),
        # mixed-precision training in the middle of a network
        _case("step_32x128x28x28_r16_bf16", STEP, 32, 128, 28, 28, 128, 3, 16, dtype="bf16"),
        # a downsampling layer on AlexNet's odd 55 x 55 plane, trained
        _case("step_16x128x55x55_r32_s2", STEP, 16, 128, 55, 55, 256, 3, 32, stride=2),
        # a network's first layer, three ragged channels in, trained: no input gradient
        _case("step_16x3x224x224_r16_first", STEP, 16, 3, 224, 224, 64, 3, 16, first=True),
        # the largest row of the all-scales list: few channels on a wide plane
        _case("fwd_16x16x512x512_r16", FORWARD, 16, 16, 512, 512, 16, 3, 16),
    ]


def _out_hw(c):
    """"same" padding: the output plane of the layer."""
    return -(-c["H"] // c["stride"]), -(-c["W"] // c["stride"])


def work(c):
    """Bytes: every input read once, every output written once.  Flops: the cheaper of the
    two orders of summation - factor by factor, or through the recomposed filter."""
    oh, ow = _out_hw(c)
    ip, op_ = c["N"] * c["H"] * c["W"], c["N"] * oh * ow
    size = DTYPES[c["dtype"]].itemsize
    x, y = size * c["C"] * ip, size * c["T"] * op_
    bias = 4 * c["T"]
    fac = 4 * c["R"] * (c["T"] + c["C"] + 2 * c["k"])
    taps = 2 * c["k"]
    dense = 2 * c["C"] * c["T"] * c["k"] ** 2 * op_
    one = min(2 * c["R"] * (c["C"] * ip + (c["T"] + taps) * op_), dense)
    grads = min(2 * c["R"] * (2 * c["C"] * ip + (2 * c["T"] + 3 * taps) * op_), dense)
    if c["op"] == INFER:
        return {"bytes": x + y + fac + bias, "flops": one}
    if c["op"] in (FORWARD, BACKWARD_DATA):
        return {"bytes": x + y + fac, "flops": one}
    if c["op"] == BACKWARD_FILTER:
        return {"bytes": x + y + 2 * fac, "flops": grads}
    dx = 0 if c["first"] else 1     # x, dy and the parameters in; y, dx and the gradients out
    return {"bytes": (1 + dx) * x + 2 * y + 2 * (fac + bias), "flops": (1 + dx) * one + grads}


def tolerance(c):
    """About four times the largest error seen against the same case evaluated in 64 bits,
    over the listed cases and 700 drawn ones (2-norm error of any output; largest single
    difference):

    * inference and the passes over activations: 3.8e-7 and 4.7e-6 in fp32 (exact products,
      sums in fp32); 1.7e-3 and 3.9e-3 in bf16, 2.2e-4 and 4.9e-4 in fp16 (the rounding of
      the stored result);
    * factor gradients in fp32: 1.8e-5 and 3.6e-5 (sums over all pixels that nearly cancel);
    * a training step: 1.2e-3 in fp32, 1.7e-3 in bf16, 2.3e-3 in fp16.  ReLU's backward
      drops dy where y = 0: for an output within rounding of zero another order of
      summation decides otherwise, and that element of dy then counts in full in every
      gradient (0.57 of dx's root mean square at one place).
    """
    if c["op"] == STEP:
        return {"rel": {"f32": 5e-3, "bf16": 7e-3, "f16": 9e-3}[c["dtype"]], "max": 0.9}
    if c["op"] == BACKWARD_FILTER:
        return {"rel": 7e-5, "max": 1.5e-4}
    return {"f32": {"rel": 1.5e-6, "max": 2e-5}, "bf16": {"rel": 7e-3, "max": 1.6e-2},
            "f16": {"rel": 9e-4, "max": 2e-3}}[c["dtype"]]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng):
    c = _log_uniform(rng, 1, 512)
    # half of them as networks have them, the others any number
    return max(16, 16 * round(c / 16)) if c > 12 and rng.random() < 0.6 else c


def draw(rng):
    limit = [work(c) for c in listed()]
    most = {k: max(w[k] for w in limit) for k in ("bytes", "flops")}
    while True:
        op = rng.choice([INFER, INFER, STEP, STEP, STEP, FORWARD, BACKWARD_DATA, BACKWARD_FILTER])
        layer = op in (INFER, STEP)
        H = _log_uniform(rng, 7, 512)
        W = H if rng.random() < 0.7 else min(512, max(7, round(H * rng.uniform(0.5, 2))))
        k = rng.choice([1, 3, 3, 3, 3, 5] + ([7] if op in (INFER, FORWARD, BACKWARD_DATA) else []))
        first = op == STEP and rng.random() < 0.15
        c = dict(op=op, N=_log_uniform(rng, 1, 128), C=3 if first else _channels(rng), H=H, W=W,
                 T=_channels(rng), k=k, R=_log_uniform(rng, 1, 64),
                 dtype=rng.choice(["f32", "f32", "bf16", "f16"]) if layer else "f32",
                 stride=1, first=first)
        if layer and c["dtype"] == "f32" and not first and rng.random() < 0.2:
            c["stride"] = 2
        w = work(c)
        if w["bytes"] >= 1 << 16 and all(w[m] <= most[m] for m in most):
            return c


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, device="cuda", generator=gen)

    dtype = DTYPES[c["dtype"]]
    N, C, H, W, T, k, R = (c[n] for n in ("N", "C", "H", "W", "T", "k", "R"))
    oh, ow = _out_hw(c)
    state = dict(case=c, pad=k // 2)
    # activations as they come: pixels in [-1, 1] at the first layer, ReLU outputs after it
    if c["op"] != BACKWARD_DATA:
        if c["first"] or C <= 4:
            x = torch.rand((N, C, H, W), device="cuda", generator=gen) * 2 - 1
        else:
            x = normal(N, C, H, W).clamp_(min=0)
        state["x"] = x.to(dtype)
    if c["op"] in (STEP, BACKWARD_DATA, BACKWARD_FILTER):
        state["dy"] = normal(N, T, oh, ow).to(dtype)
    # factors of the layer's own initial scale: the recomposed filter is Kaiming-normal
    scale = (2.0 / (C * k * k * R)) ** 0.125
    factors = [normal(d, R) * scale for d in (T, C, k, k)]
    if c["op"] not in (INFER, STEP):
        state["factors"] = factors
        return state
    layer = torch_ops.CP4Conv2d(C, T, k, R, bias=True, activation="relu", stride=c["stride"],
                                padding="same")
    with torch.no_grad():
        for p, f in zip((layer.FK, layer.FC, layer.FH, layer.FW), factors):
            p.copy_(f)
        layer.bias.copy_(0.1 * normal(T))
    state["layer"] = layer
    if c["op"] == STEP and not c["first"]:
        state["x"].requires_grad_()
    return state


def run(state):
    c = state["case"]
    if c["op"] == INFER:
        with torch.no_grad():
            return state["layer"](state["x"])
    if c["op"] == STEP:
        x, layer = state["x"], state["layer"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(state["dy"])
        out = {"y": y.detach(), "bias": layer.bias.grad, "FK": layer.FK.grad,
               "FC": layer.FC.grad, "FH": layer.FH.grad, "FW": layer.FW.grad}
        if not c["first"]:
            out["x"] = x.grad
        return out
    if c["op"] == FORWARD:
        return cp4.conv2d_forward(state["x"], *state["factors"], pad=state["pad"])
    if c["op"] == BACKWARD_DATA:
        return cp4.conv2d_backward_data(state["dy"], *state["factors"], pad=state["pad"])
    return cp4.conv2d_backward_filter(state["x"], state["dy"], *state["factors"],
                                      pad=state["pad"])
