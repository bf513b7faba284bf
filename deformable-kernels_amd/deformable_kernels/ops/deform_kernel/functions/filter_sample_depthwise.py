"""The two depthwise deformable-kernel operators with their gradients.

Same call signatures, tensor layouts and gradient set as the reference's
``SampleDepthwiseFunction`` and ``DeformableSampleDepthwiseFunction``
(``functions/filter_sample_depthwise.py:19-102`` and ``:105-206``); the autograd
nodes are native code (``csrc/dk_torch.cpp``) over the C ABI of ``libdk_hip.so``.

Differences a user can observe:
  * ``backward`` returns one gradient slot per forward argument (the
    reference returns one too few -- ``:87`` and ``:191`` -- which current
    PyTorch rejects);
  * tensors are validated (device, dtype, shape) and a failing native call
    raises instead of printing;
  * bfloat16 is accepted; fp16/bf16 accumulate in fp32;
  * one optional trailing argument, ``rotation_clip`` (``None``, a ``(min, max)`` pair or
    ``'scope'``): the clamp the reference's module applies to the rotation tensor before the
    call (``modules/deform_kernel.py:185-212``), applied inside the kernels instead;
  * a channels-last input gets a channels-last output and channels-last gradients;
  * ``rotation = None`` in the deformable operator: no kernel-space offsets, the library reads no tensor of zeros;
  * the ``apex.amp.float_function`` wrapper (``:209-211``) is replaced by an
    autocast-aware cast to fp32, apex not being a dependency.
"""
import torch

from .. import _lib

__all__ = ['sample_depthwise', 'deform_sample_depthwise']


class SampleDepthwiseFunction:
    """``SampleDepthwiseFunction.apply`` of the reference (``:19-102``)."""

    @staticmethod
    def apply(input, rotation, weight, kernel_size=(3, 3), stride=(1, 1), padding=(1, 1), dilation=(1, 1),
              rotation_groups=1, rotation_clip=None):
        return _lib.native().sample_depthwise(
            input, rotation, weight, kernel_size, stride, padding, dilation, rotation_groups,
            *_lib.clip_triple(rotation_clip, weight))


class DeformableSampleDepthwiseFunction:
    """``DeformableSampleDepthwiseFunction.apply`` of the reference (``:105-206``)."""

    @staticmethod
    def apply(input, offset, rotation, weight, kernel_size=(3, 3), stride=(1, 1), padding=(1, 1), dilation=(1, 1),
              rotation_groups=1, rotation_clip=None):
        return _lib.native().deform_sample_depthwise(
            input, offset, rotation, weight, kernel_size, stride, padding, dilation, rotation_groups,
            *_lib.clip_triple(rotation_clip, weight))


def _float_function(fn):
    """Stand-in for ``apex.amp.float_function`` (reference ``:209-211``): inside an
    autocast region the floating-point tensor arguments are cast to fp32 and the
    op runs with autocast off; outside one it is the identity wrapper."""
    def wrapper(*args):
        if torch.is_autocast_enabled():
            args = tuple(a.float() if torch.is_tensor(a) and a.is_floating_point() else a for a in args)
            with torch.autocast(device_type="cuda", enabled=False):
                return fn(*args)
        return fn(*args)
    wrapper.__wrapped__ = fn
    return wrapper


# register as fp32 functions.
sample_depthwise = _float_function(SampleDepthwiseFunction.apply)
deform_sample_depthwise = _float_function(DeformableSampleDepthwiseFunction.apply)
