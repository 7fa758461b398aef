"""Grouped (depthwise) causal conv1d + activation: ``GroupedConv1dNKI`` / ``nki_conv1d`` /
``ConvNKI`` with the reference's signatures (``mamba2/conv1d_grouped.py:265-334``), computed by
the gfx950 HIP kernels.

Layout: the reference module takes (B, C, L) (``:300-306``); the mixer's fused path uses the
sequence-major (B, L, C) layout (``:66-125``).  Both are supported here: ``channels_last=False``
(default, reference layout) or ``True``.  weight is (C, 1, k), bias (C) or None.
"""
from typing import Union

import torch
import torch.nn as nn

from . import _lib


def _activation_code(activation):
    if activation not in _lib.ACT:
        raise ValueError(f"Invalid activation {activation}")
    return _lib.ACT[activation]


def conv1d_forward(input, weight, bias=None, activation=None, channels_last=False, out=None):
    return _lib.native().conv1d_forward(input, weight, bias, _activation_code(activation), channels_last, out)


def conv1d_backward(input, weight, bias, d_output, activation=None, channels_last=False, out_dx=None):
    return _lib.native().conv1d_backward(input, weight, bias, d_output, _activation_code(activation), channels_last, out_dx)


class GroupedConv1dNKI(torch.autograd.Function):
    """apply(input, weight, bias, activation=None) -> output;
    backward -> (dinput, dweight, dbias, None)   (``conv1d_grouped.py:267,279,288``).  The node itself is C++
    (csrc/binding.cpp)."""

    @staticmethod
    def apply(input, weight, bias, activation=None, channels_last=False):
        return _lib.native().conv1d(input, weight, bias, _activation_code(activation), channels_last)


def nki_conv1d(input, weight, bias=None, activation=None, channels_last=False):
    return GroupedConv1dNKI.apply(input, weight, bias, activation, channels_last)


class ConvNKI(nn.Conv1d):
    """Depthwise causal conv layer equivalent to ``nn.Conv1d(C, C, k, groups=C, padding=k-1)(x)[..., :L]``
    followed by ``activation``.  input (B, C, L), weight (C, 1, k), bias (C)  (``conv1d_grouped.py:295-334``).
    The tensor-parallel slicing of the reference (``:323-331``) is the identity on one GPU."""

    def __init__(self, in_channels: int, out_channels: int, kernel_size: int, stride: int = 1,
                 padding: Union[str, int] = 0, dilation: int = 1, groups: int = 1, bias: bool = True,
                 padding_mode: str = 'zeros', device=None, dtype=None, activation=None) -> None:
        assert groups == in_channels, "grouped conv kernel only supports groups == in_channels"
        assert padding == kernel_size - 1
        assert padding_mode == 'zeros'
        assert dilation == 1
        assert stride == 1
        super().__init__(in_channels, out_channels, kernel_size, stride, padding, dilation, groups, bias, padding_mode,
                         device, dtype)
        self.activation = activation

    def forward(self, input):
        return GroupedConv1dNKI.apply(input, self.weight, self.bias, self.activation, False)
