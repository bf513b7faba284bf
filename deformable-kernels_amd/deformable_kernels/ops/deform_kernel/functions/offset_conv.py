"""The offset branch of ``LocalDeformKernel2d``: its 3x3 ``rotation_conv`` (reference
``modules/deform_kernel.py:165-168``, applied at ``:214``).

``offset_conv(input, weight, bias, stride, padding, dilation)`` returns what
``torch.nn.functional.conv2d`` returns.  For float32, float16 and bfloat16 GPU tensors (all of one dtype; fp32
sums, results rounded once) with padding 1, dilation 1, input channels a multiple of 16 (16-bit tensors: any number,
with the forward on the framework's routine unless ``force=True``), 18 output channels or at most 16, on planes 7, 14, 28, 56 or 112 wide (stride 2: input planes 14 to 112 wide) it runs

  * the forward and the input gradient on the library's shift-GEMM kernels on the 16-bit matrix instructions:
    float16 / bfloat16 elements as they are (exact products), float32 elements as bfloat16 (hi, lo) pairs
    (about 3.5e-6 of the result's scale against the float64 convolution),
  * the weight gradient on the library's kernel for the 16-bit matrix instructions (stride 1 and 2, up to 20
    outputs; float32 tensors again as bfloat16 pairs), per-workgroup partial sums added in a fixed order,
  * the bias gradient on the library's reduction kernel for every shape (the framework's
    reduction over (N, H, W) takes 60-230 us on the large planes),
  * of these shapes, most of those with too few images to fill the GPU that way (up to 2 M output pixels times input
    channels, at stride 2 0.6 M for the gradients; the queries ``dk_offset_conv_direct_worthwhile`` and
    ``dk_offset_conv_direct_backward_worthwhile`` tell), and the gradients of 16-bit tensors with other channel counts and on other
    planes up to 0.6 M (stride 2 0.37 M): one fp32 vector-unit kernel per pass (``csrc/dk_offset_direct.hip``),
  * everything else -- other shapes, and passes the library reports as covered
    but not worthwhile (the float32 input gradient with fewer than 64 channels or
    on 7 x 7 planes; few images of many channels) unless ``force=True`` -- on the framework's convolution routines.

float64, CPU tensors, mixed dtypes and autocast regions go to ``F.conv2d`` unchanged.  The autograd node is native code
(``csrc/dk_torch.cpp``).
"""
import torch
import torch.nn.functional as F

from .. import _lib

__all__ = ['offset_conv', 'offset_conv_supported']


_NATIVE_DTYPES = (torch.float32, torch.float16, torch.bfloat16)


def _pair(v):
    """Both dimensions' value of a convolution argument: a number, a pair, or (as F.conv2d takes) one number in a list."""
    if isinstance(v, (tuple, list)):
        return tuple(int(e) for e in v) if len(v) != 1 else (int(v[0]), int(v[0]))
    return int(v), int(v)


def offset_conv_supported(input, weight, bias, stride, padding, dilation, worthwhile=False):
    """Whether the native forward / weight-gradient kernels cover this call; with ``worthwhile``
    also whether they are expected to be faster than the library convolution."""
    if torch.is_autocast_enabled():
        return False
    return _lib.native().offset_conv_supported(input, weight, bias, _pair(stride), _pair(padding), _pair(dilation),
                                               bool(worthwhile))


def offset_conv(input, weight, bias=None, stride=1, padding=1, dilation=1, force=False):
    """``F.conv2d(input, weight, bias, stride, padding, dilation)`` for the offset branch (see the
    module docstring for what runs where)."""
    if (not input.is_cuda or torch.is_autocast_enabled()
            or isinstance(padding, str) and input.dtype not in _NATIVE_DTYPES):
        return F.conv2d(input, weight, bias, stride, padding, dilation)
    return _lib.native().offset_conv(input, weight, bias, _pair(stride), _pair(padding), _pair(dilation), bool(force))
