"""PyTorch autograd binding of the fused CP4 Conv2d C ABI.

Stands where the reference registers its TensorFlow custom op
(Kernels/cp4_conv_nchw.cc:6-108, ``Cp4Conv2dNchw``: input + four factor
tensors -> output, NCHW): a ``torch.autograd.Function`` whose forward, input
gradient and factor gradients are the three passes of ``libcp4conv.so``.
PyTorch only owns the tensors and the stream; all arithmetic is in the HIP
library, and there is no eager fallback.

Factor layout is the C ABI's: FK [T,R], FC [C,R], FH [Y,R], FW [X,R].
For "same" padding at stride 1 (2*pad = Y-1 = X-1) the reference's three passes
run as they are; that is the only case in which its backward-data formula
(flipped taps at offset +y-pad, Cuda_kernels/cp4Conv2dBackwardData.cu:79-87) is
the adjoint of its forward.  Strides and every other padding go through the
library's geometry entry points (cp4_conv2d_forward_ex and its exact gradients).

Launches are asynchronous.  A producer / consumer kernel whose wait between waves
runs out ends early and leaves its output incomplete; the library records that per
device and reports it from ``cp4_device_status``, which synchronises the stream.
``check_device()`` is that call: use it wherever the training loop synchronises
anyway (reading the loss, a checkpoint).  ``set_device_checks(True)`` - or the
environment variable ``CP4_CHECK_DEVICE=1`` - makes every backward pass of the
Functions below end with it, at the price of one synchronisation per layer and step.
"""
import os

import torch

from . import capi


def set_device_checks(on):
    """Check the device's fault record at the end of every backward pass (synchronises)."""
    global _check_every_backward
    _check_every_backward = bool(on)
    if not isinstance(capi._native, capi._Missing):
        capi._native.set_check_backward(_check_every_backward)


set_device_checks(os.environ.get("CP4_CHECK_DEVICE", "0") not in ("", "0"))


def check_device(stream=None):
    """Synchronises ``stream`` and raises ``capi.Cp4Error`` (ERR_DEVICE) if a kernel of
    the library gave up a wait since the last check: outputs computed since then are
    incomplete.  The record is cleared."""
    capi.device_status(stream)


def _after_backward():
    if _check_every_backward:
        capi.device_status()


class CP4Conv2dFunction(torch.autograd.Function):
    """y = act(cp4conv2d(x, FK, FC, FH, FW, pad) + bias) as a Python autograd function, forward
    and backward each one call of the library's layer entry points.  ``cp4_conv2d`` runs the
    native one (csrc/torch/binding.cpp); this one stands for it where a call has to be seen
    as an operator: in a trace.

    A bfloat16 or float16 ``x`` selects the library's 16-bit activations (y and the input
    gradient are of x's type then; factors, bias and their gradients stay float32); shapes
    those do not take run on widened copies.
    """

    @staticmethod
    def forward(ctx, x, FK, FC, FH, FW, pad, bias=None, activation=None):
        if 2 * pad + 1 != FH.shape[0] or 2 * pad + 1 != FW.shape[0]:
            raise ValueError("autograd binding needs 2*pad = Y-1 = X-1 (the reference's "
                             "backward-data pass is the adjoint only then)")
        x = x.contiguous()
        if x.dtype not in (torch.bfloat16, torch.float16):
            x = x.float()
        return _layer_forward(ctx, x, FK, FC, FH, FW, pad, None, bias, activation)

    @staticmethod
    def backward(ctx, dy):
        return _layer_backward(ctx, dy)


class CP4Conv2dGeometryFunction(torch.autograd.Function):
    """The same for a layer with a stride, explicit padding or an output plane of its own
    (``geom``: a ``capi.Geometry``; float32)."""

    @staticmethod
    def forward(ctx, x, FK, FC, FH, FW, geom, bias=None, activation=None):
        return _layer_forward(ctx, x.contiguous().float(), FK, FC, FH, FW, 0, geom, bias,
                              activation)

    @staticmethod
    def backward(ctx, dy):
        return _layer_backward(ctx, dy)


def _layer_forward(ctx, x, FK, FC, FH, FW, pad, geom, bias, activation):
    FK, FC, FH, FW = (t.contiguous().float() for t in (FK, FC, FH, FW))
    if bias is not None:
        bias = bias.contiguous().float()
    s = capi.shape_for(x.shape, FK, FC, FH, FW, pad)
    y = capi.layer_forward(s, geom, x, FK, FC, FH, FW, bias, activation)
    ctx.shape, ctx.geom, ctx.activation = s, geom, activation
    ctx.save_for_backward(x, FK, FC, FH, FW, y if capi.ACTIVATIONS[activation] == 1 else None)
    return y


def _layer_backward(ctx, dy):
    x, FK, FC, FH, FW, y = ctx.saved_tensors
    need = ctx.needs_input_grad
    # create_graph: the bias gradient is linear in dy and stays differentiable
    bias_graph = need[6] and torch.is_grad_enabled() and dy.requires_grad
    dx, grads, dbias = capi.layer_backward(
        ctx.shape, ctx.geom, x, y, dy.contiguous().to(x.dtype), FK, FC, FH, FW, ctx.activation,
        want_dx=need[0], want_factors=any(need[1:5]), want_bias=need[6] and not bias_graph)
    if bias_graph:
        dbias = (dy if y is None else dy * (y > 0)).float().sum(dim=(0, 2, 3))
    grads = tuple(g if n else None for g, n in zip(grads, need[1:5]))
    _after_backward()
    return (dx,) + grads + (None, dbias, None)


def _traced_layer(x, FK, FC, FH, FW, pad, bias, activation, stride, padding):
    if padding is None:
        padding = pad
    y_taps, x_taps = FH.shape[0], FW.shape[0]
    if stride == 1 and (
            (isinstance(padding, int) and 2 * padding + 1 == y_taps == x_taps) or
            (padding == "same" and y_taps == x_taps and y_taps % 2 == 1)):
        return CP4Conv2dFunction.apply(x, FK, FC, FH, FW, y_taps // 2, bias, activation)
    geom = capi.geometry(capi.shape_for(x.shape, FK, FC, FH, FW, 0), stride, padding)
    return CP4Conv2dGeometryFunction.apply(x, FK, FC, FH, FW, geom, bias, activation)


def cp4_conv2d(x, FK, FC, FH, FW, pad, bias=None, activation=None, stride=1, padding=None):
    """Functional form: differentiable fused CP4 convolution (NCHW), with the
    optional bias [T] and activation ("relu") fused into the forward stores.

    ``pad`` zeros on every side, stride 1 and 2*pad = Y - 1 is the reference's own
    layer and runs its three passes (bfloat16 activations included).  A ``stride``,
    ``padding`` = "same" (the framework's rule of the reference's Python layers,
    test/layers.py:264-279: out = ceil(in / stride), on even sizes one more zero
    after the image than before it), "valid", an int or an (h, w) pair run the
    strided kernels: only the kept outputs are computed.
    """
    # torch.jit.trace records operators: the native call would leave a constant in the graph
    run = capi._native.layer if torch._C._get_tracing_state() is None else _traced_layer
    return run(x, FK, FC, FH, FW, pad, bias, activation, stride, padding)


class CP4Conv2d(torch.nn.Module):
    """A rank-R CP4-decomposed convolution layer, "same" padding.

    Equivalent dense filter: K[t,c,y,x] = sum_r FK[t,r] FC[c,r] FH[y,r] FW[x,r]
    (Cuda_kernels/Utils.cu:55-62).  Factors start as normal(0, s) with s chosen
    so that the recomposed filter has the variance of a Kaiming-normal dense
    filter of the same shape.
    """

    def __init__(self, in_channels, out_channels, kernel_size, rank, device="cuda", bias=False,
                 activation=None, stride=1, padding=None):
        super().__init__()
        if kernel_size % 2 != 1 and padding is None:
            raise ValueError("kernel_size must be odd for the default padding")
        self.pad = kernel_size // 2
        self.padding = padding
        fan_in = in_channels * kernel_size * kernel_size
        # Var[K] = R * s^8 for four independent N(0, s^2) factors; target 2 / fan_in
        s = (2.0 / (fan_in * rank)) ** 0.125
        mk = lambda d: torch.nn.Parameter(torch.randn(d, rank, device=device) * s)
        self.FK, self.FC = mk(out_channels), mk(in_channels)
        self.FH, self.FW = mk(kernel_size), mk(kernel_size)
        self.bias = torch.nn.Parameter(torch.zeros(out_channels, device=device)) if bias else None
        self.activation = activation
        self.stride = stride

    def forward(self, x):
        return cp4_conv2d(x, self.FK, self.FC, self.FH, self.FW, self.pad, self.bias,
                          self.activation, self.stride, self.padding)

    @staticmethod
    def check_device(stream=None):
        """See ``check_device``: call where the loop synchronises anyway."""
        check_device(stream)

    def dense_filter(self):
        """The recomposed [T,C,Y,X] filter (on the device, through cp4_recompose)."""
        return capi.recompose(self.FK.detach(), self.FC.detach(), self.FH.detach(),
                              self.FW.detach())


class CP3Conv2dFunction(torch.autograd.Function):
    """The 3-factor CP convolution of the reference's ``Conv2dCpFusedNchw`` op
    (Kernels/cp_fused_nchw.cc:6-30; its Python definition is pointwise K0,
    depthwise K1, pointwise K2, test/layers.py:265-282):

        y[n,t] = sum_r K2[r,t] * (K1[:,:,r] (*) sum_c K0[c,r] x[n,c])

    K0 [C,R], K1 [Y,X,R], K2 [R,T].  All three passes are the library's cp3 entry
    points.
    """

    @staticmethod
    def forward(ctx, x, K0, K1, K2, pad):
        if 2 * pad + 1 != K1.shape[0] or 2 * pad + 1 != K1.shape[1]:
            raise ValueError("autograd binding needs 2*pad = Y-1 = X-1")
        K0, K1, K2 = (t.contiguous().float() for t in (K0, K1, K2))
        x = x.contiguous().float()
        ctx.pad = pad
        ctx.save_for_backward(x, K0, K1, K2)
        return capi.cp3_conv2d_forward(x, K0, K1, K2, pad=pad)

    @staticmethod
    def backward(ctx, dy):
        x, K0, K1, K2 = ctx.saved_tensors
        dy = dy.contiguous().float()
        dx = None
        if ctx.needs_input_grad[0]:
            dx = capi.cp3_conv2d_backward_data(dy, K0, K1, K2, pad=ctx.pad)
        grads = (None, None, None)
        if any(ctx.needs_input_grad[1:4]):
            grads = capi.cp3_conv2d_backward_filter(x, dy, K0, K1, K2, pad=ctx.pad)
            grads = tuple(g if need else None for g, need in zip(grads, ctx.needs_input_grad[1:4]))
        _after_backward()
        return (dx,) + grads + (None,)


def cp3_conv2d(x, K0, K1, K2, pad):
    """Functional form of the differentiable 3-factor CP convolution (NCHW)."""
    return CP3Conv2dFunction.apply(x, K0, K1, K2, pad)


class CP3Conv2d(torch.nn.Module):
    """A rank-R 3-factor CP convolution layer, "same" padding: pointwise K0 [C,R],
    depthwise K1 [k,k,R], pointwise K2 [R,T] (the kernels of the reference's Python
    layer, test/layers.py:285-294, in the fused op's layouts).  Factors start as
    normal(0, s) with s chosen so that the equivalent dense filter
    sum_r K0[c,r] K1[i,j,r] K2[r,t] has the variance of a Kaiming-normal one."""

    def __init__(self, in_channels, out_channels, kernel_size, rank, device="cuda"):
        super().__init__()
        if kernel_size % 2 != 1:
            raise ValueError("kernel_size must be odd (same padding)")
        self.pad = kernel_size // 2
        fan_in = in_channels * kernel_size * kernel_size
        # Var = R * s^6 for three independent N(0, s^2) factors; target 2 / fan_in
        s = (2.0 / (fan_in * rank)) ** (1.0 / 6.0)
        mk = lambda *d: torch.nn.Parameter(torch.randn(*d, device=device) * s)
        self.K0 = mk(in_channels, rank)
        self.K1 = mk(kernel_size, kernel_size, rank)
        self.K2 = mk(rank, out_channels)

    def forward(self, x):
        return cp3_conv2d(x, self.K0, self.K1, self.K2, self.pad)


class RCPConv2dFunction(torch.autograd.Function):
    """The reshaped-CP convolution of the reference's ``Conv2dRcpFusedNchw`` op
    (Kernels/rcp_fused_nchw.cc:6-12; test/test_conv2d_rcp.py:38-41):

        y[n,(x,y)] = sum_r sum_{a,b} K0[a,x,r] K1[b,y,r] * (KC[:,:,r] (*) x[n,(a,b)])

    K0 [S0,T0,R], K1 [S1,T1,R], KC [Y,X,R]; x has S0*S1 channels, y T0*T1.  All three
    passes are the library's rcp entry points."""

    @staticmethod
    def forward(ctx, x, K0, K1, KC, pad):
        if 2 * pad + 1 != KC.shape[0] or 2 * pad + 1 != KC.shape[1]:
            raise ValueError("autograd binding needs 2*pad = Y-1 = X-1")
        K0, K1, KC = (t.contiguous().float() for t in (K0, K1, KC))
        x = x.contiguous().float()
        ctx.pad = pad
        ctx.save_for_backward(x, K0, K1, KC)
        return capi.rcp_conv2d_forward(x, K0, K1, KC, pad=pad)

    @staticmethod
    def backward(ctx, dy):
        x, K0, K1, KC = ctx.saved_tensors
        dy = dy.contiguous().float()
        dx = None
        if ctx.needs_input_grad[0]:
            dx = capi.rcp_conv2d_backward_data(dy, K0, K1, KC, pad=ctx.pad)
        grads = (None, None, None)
        if any(ctx.needs_input_grad[1:4]):
            grads = capi.rcp_conv2d_backward_filter(x, dy, K0, K1, KC, pad=ctx.pad)
            grads = tuple(g if need else None for g, need in zip(grads, ctx.needs_input_grad[1:4]))
        _after_backward()
        return (dx,) + grads + (None,)


def rcp_conv2d(x, K0, K1, KC, pad):
    """Functional form of the differentiable reshaped-CP convolution (NCHW)."""
    return RCPConv2dFunction.apply(x, K0, K1, KC, pad)
