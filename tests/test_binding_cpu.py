"""The binding's argument handling, as far as it goes before a device is needed: what it
takes ends at the check for device tensors, what it refuses ends earlier with its own error."""
import numpy as np
import pytest
import torch

from paralleltnnlayers_amd import torch_ops


def _layer(stride=1, padding=None, taps=3):
    x, fac = torch.zeros(1, 4, 9, 9), [torch.zeros(d, 2) for d in (6, 4, taps, taps)]
    return torch_ops.cp4_conv2d(x, *fac, taps // 2, stride=stride, padding=padding)


# (the plain layer takes whatever equals 1, as `stride == 1` does)
@pytest.mark.parametrize("stride", [1, True, 1.0, np.int64(1), np.float32(1), (1, 1), 2, (2, 1),
                                    [np.int64(2), 2]], ids=repr)
def test_stride_forms_that_are_taken(stride):
    with pytest.raises(AssertionError, match="device tensor"):
        _layer(stride)


@pytest.mark.parametrize("stride,padding", [(np.int64(2), None), (2.0, None), (1.0, "valid"),
                                            (np.int64(1), (1, 1)), ("1", None)], ids=repr)
def test_stride_forms_that_are_refused(stride, padding):
    with pytest.raises((TypeError, ValueError)):
        _layer(stride, padding)


def _pass(name, *fac):
    from paralleltnnlayers_amd import capi
    x, dy = torch.zeros(1, 4, 5, 5), torch.zeros(1, 6, 5, 5)

    class Stream:               # (without a device there is no current one to ask for)
        cuda_stream = 0

    if name == "conv2d_forward":
        return capi._native.forward(x, *fac, 1, None, -1, Stream)
    if name == "conv2d_backward_data":
        return capi._native.backward_data(dy, *fac, 1, None, Stream)
    if name == "conv2d_backward_filter":
        return capi._native.backward_filter(x, dy, *fac, 1, None, Stream, -1)
    return torch_ops.cp4_conv2d(x, *fac, 1)


PASSES = ["conv2d_forward", "conv2d_backward_data", "conv2d_backward_filter", "layer"]


@pytest.mark.parametrize("forms", [((6, 2), (4, 2), (3, 2), (3, 2)), ((6, 1), (4, 1), (3,), (3,)),
                                   ((6, 2, 1), (4, 2), (3, 2, 1), (3, 1, 2)), ((6, 1), (4,), (3,), (3, 1))],
                         ids=repr)
@pytest.mark.parametrize("name", PASSES)
def test_factor_forms_that_are_taken(name, forms):
    """Rows and rank count; FC names its channels by its second dimension only in the backward
    passes."""
    refused = len(forms[1]) == 1 and name in ("conv2d_forward", "layer")
    with pytest.raises(AssertionError, match="match" if refused else "device tensor"):
        _pass(name, *[torch.zeros(*f) for f in forms])


@pytest.mark.parametrize("short", [1, 2, 3])
@pytest.mark.parametrize("name", PASSES)
def test_factors_with_too_few_entries_are_refused(name, short):
    """The kernels would read past their end."""
    fac = [torch.zeros(d, 2) for d in (6, 4, 3, 3)]
    fac[short] = fac[short][:, :1].contiguous()
    with pytest.raises(AssertionError, match="fewer"):
        _pass(name, *fac)


class _OnDevice(torch.Tensor):
    """A host tensor that says it is on the device."""
    is_cuda = True


class _Reached(Exception):
    pass


@pytest.fixture()
def layer_calls(monkeypatch):
    """capi's layer functions down to the library call, which raises _Reached."""
    from paralleltnnlayers_amd import capi

    class Lib:
        def __getattr__(self, name):
            def call(*args):
                if name.endswith("workspace_bytes"):
                    return 0
                raise _Reached(name)
            return call

    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **k).as_subclass(_OnDevice))
    monkeypatch.setattr(capi, "lib", lambda: Lib())
    monkeypatch.setattr(capi, "_stream", lambda stream: None)
    return capi


def _on_device(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype).as_subclass(_OnDevice)


@pytest.mark.parametrize("fault", [None, "dy type", "dy shape", "y type", "y shape", "x shape", "FH",
                                   "bias"])
def test_layer_calls_check_types_and_sizes(layer_calls, fault):
    """An operand of another type or size than the layer's never reaches the library, whose
    kernels would read past its end."""
    capi = layer_calls
    f32, bf16 = torch.float32, torch.bfloat16
    x = _on_device(2, 4, 5, 7)
    y = _on_device(2, 6, 5, 7 if fault != "y shape" else 6, dtype=bf16 if fault == "y type" else f32)
    dy = _on_device(2, 6, 5, 7 if fault != "dy shape" else 6, dtype=bf16 if fault == "dy type" else f32)
    fac = [_on_device(6, 3), _on_device(4, 3), _on_device(3, 2 if fault == "FH" else 3), _on_device(3, 3)]
    s = capi.shape_for(x.shape, *fac, 1)
    if fault == "x shape":
        x = _on_device(2, 3, 5, 7)
    backward = lambda: capi.layer_backward(s, None, x, y, dy, *fac, "relu", want_bias=False)
    with pytest.raises(_Reached if fault in (None, "bias") else AssertionError):
        backward()
    if fault in ("dy type", "dy shape", "y type", "y shape"):
        return
    bias = _on_device(6 if fault != "bias" else 5)
    with pytest.raises(_Reached if fault is None else AssertionError):
        capi.layer_forward(s, None, x, *fac, bias, "relu")
