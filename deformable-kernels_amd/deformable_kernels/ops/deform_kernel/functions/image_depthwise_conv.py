"""The convolution ``GlobalDeformKernel2d`` applies with its per-image kernels (reference
``modules/deform_kernel.py:103-111``): ``F.conv2d(x.view(1, n * c, h, w), weight, groups = n * c)``
for a depthwise layer, where ``weight`` holds one ``k x k`` kernel per image and channel.

``image_depthwise_conv(input, weight, stride, padding, dilation)`` takes ``input`` as
``[N, C, H, W]`` and ``weight`` as ``[N * C, 1, k_h, k_w]`` (what ``dynamic_weight`` returns) or
``[N, C, k_h, k_w]`` -- the latter in any dense layout, in particular the permuted view of the
sampler's ``[N * k_h * k_w, C]`` output, which saves the transposing copy of ``:97-101`` and its
gradient -- and returns ``[N, C, H_out, W_out]``: the values and gradients of that grouped
convolution, computed by the library's streaming kernels (forward, input gradient, kernel
gradient; ``include/dk_hip.h``: ``dk_image_depthwise_*``).  GPU tensors only; geometries the
kernels do not cover (``image_depthwise_conv_supported``) are the caller's to route to ``F.conv2d``.
The autograd node is native code (``csrc/dk_torch.cpp``).
"""
from .. import _lib

__all__ = ['image_depthwise_conv', 'image_depthwise_conv_supported']


def _pair(v):
    return tuple(int(e) for e in v) if isinstance(v, (tuple, list)) else (int(v), int(v))


def _desc(input, k_h, k_w, stride, padding, dilation):
    return _lib.ConvDesc(
        input.size(0), input.size(1), input.size(2), input.size(3), k_h, k_w, stride[0], stride[1],
        padding[0], padding[1], dilation[0], dilation[1], 1, 1, 1, _lib.dtype_tag(input), _lib.CLIP_NONE, 0.0, 0.0)


def image_depthwise_conv_supported(input, weight, stride=1, padding=0, dilation=1):
    """Whether the library's kernels cover this call (GPU tensors of one dtype, a geometry whose
    taps fit the kernels' staging area)."""
    if not (input.is_cuda and weight.is_cuda and input.dtype == weight.dtype and input.dtype in _lib._DTYPES):
        return False
    if input.dim() != 4 or weight.dim() != 4:
        return False
    desc = _desc(input, weight.size(2), weight.size(3), _pair(stride), _pair(padding), _pair(dilation))
    return bool(_lib.lib().dk_image_depthwise_supported(desc))


def image_depthwise_conv(input, weight, stride=1, padding=0, dilation=1):
    return _lib.native().image_depthwise_conv(input, weight, _pair(stride), _pair(padding), _pair(dilation))
