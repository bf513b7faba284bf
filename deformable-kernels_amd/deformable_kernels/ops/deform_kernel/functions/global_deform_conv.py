"""``GlobalDeformKernel2d`` of a depthwise layer as one autograd Function (reference
``modules/deform_kernel.py:68-118``): the pooled input, its linear layer, the clamped coordinates and the kernels
sampled from the scope weights for every image (``include/dk_hip.h``: ``dk_global_kernels_*``), then the per-image
depthwise convolution (``dk_image_depthwise_*``).  Values and gradients of the reference's sequence of framework
operators, each tensor that sequence rounds rounded in the same place on the way forward; on the way back the
coordinates' share of the input gradient is added before the rounding instead of after it.  The autograd node is native code (``csrc/dk_torch.cpp``).
"""
from .. import _lib

__all__ = ['global_deform_conv', 'global_deform_conv_supported']


def _pair(v):
    return tuple(int(e) for e in v) if isinstance(v, (tuple, list)) else (int(v), int(v))


def global_deform_conv_supported(input, weight, fc_weight, fc_bias, kernel_size, stride=1, padding=0, dilation=1):
    """Whether the library's kernels cover the call: GPU tensors of one dtype (not float64), ``weight``
    ``[C, 1, S_h, S_w]``, ``fc_weight`` ``[2 k k, C]``, and a geometry of the per-image convolution."""
    return _lib.native().global_deform_conv_supported(input, weight, fc_weight, fc_bias, kernel_size, _pair(stride),
                                                      _pair(padding), _pair(dilation))


def global_deform_conv(input, weight, fc_weight, fc_bias, kernel_size, stride=1, padding=0, dilation=1):
    return _lib.native().global_deform_conv(input, weight, fc_weight, fc_bias, kernel_size, _pair(stride),
                                            _pair(padding), _pair(dilation))
