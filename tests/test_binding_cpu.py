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
