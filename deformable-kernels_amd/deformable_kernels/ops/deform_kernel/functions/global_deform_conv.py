"""``GlobalDeformKernel2d`` of a depthwise layer as one autograd Function (reference
``modules/deform_kernel.py:68-118``): the pooled input, its linear layer, the clamped coordinates and the kernels
sampled from the scope weights for every image (``include/dk_hip.h``: ``dk_global_kernels_*``), then the per-image
depthwise convolution (``dk_image_depthwise_*``).  Values and gradients of the reference's sequence of framework
operators, each tensor that sequence rounds rounded in the same place on the way forward; on the way back the
coordinates' share of the input gradient is added before the rounding instead of after it.
"""
import ctypes

import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable

from .. import _lib

__all__ = ['global_deform_conv', 'global_deform_conv_supported']


def _desc(input, weight, kernel_size, stride, padding, dilation):
    return _lib.ConvDesc(
        input.size(0), input.size(1), input.size(2), input.size(3), kernel_size, kernel_size, stride[0], stride[1],
        padding[0], padding[1], dilation[0], dilation[1], weight.size(2), weight.size(3), 1, _lib.dtype_tag(input),
        _lib.CLIP_NONE, 0.0, 0.0)


def _pair(v):
    return tuple(int(e) for e in v) if isinstance(v, (tuple, list)) else (int(v), int(v))


def global_deform_conv_supported(input, weight, fc_weight, fc_bias, kernel_size, stride=1, padding=0, dilation=1):
    """Whether the library's kernels cover the call: GPU tensors of one dtype (not float64), ``weight``
    ``[C, 1, S_h, S_w]``, ``fc_weight`` ``[2 k k, C]``, and a geometry of the per-image convolution."""
    tensors = (input, weight, fc_weight, fc_bias)
    if any(t is None or not t.is_cuda or t.dtype != input.dtype or t.device != input.device for t in tensors):
        return False
    if input.dtype not in _lib._DTYPES or input.dim() != 4 or weight.dim() != 4 or input.size(0) == 0:
        return False
    if weight.size(0) != input.size(1) or weight.size(1) != 1 or \
            tuple(fc_weight.shape) != (2 * kernel_size * kernel_size, input.size(1)):
        return False
    desc = _desc(input, weight, kernel_size, _pair(stride), _pair(padding), _pair(dilation))
    L = _lib.lib()
    return bool(L.dk_global_kernels_supported(desc)) and bool(L.dk_image_depthwise_supported(desc))


class GlobalDeformConvFunction(Function):
    @staticmethod
    def forward(ctx, input, weight, fc_weight, fc_bias, kernel_size, stride, padding, dilation):
        input, weight, fc_weight, fc_bias = (t.contiguous() for t in (input, weight, fc_weight, fc_bias))
        n, c = input.size(0), input.size(1)
        taps = kernel_size * kernel_size
        desc = _desc(input, weight, kernel_size, stride, padding, dilation)
        L = _lib.lib()
        oh, ow = ctypes.c_int32(0), ctypes.c_int32(0)
        _lib.check(L.dk_conv_out_size(desc, ctypes.byref(oh), ctypes.byref(ow)), "global_deform_conv shape")
        pooled = input.new_empty(n, c)
        coord = input.new_empty(2, n, taps, 2)   # as predicted, and clamped to the scope
        kernels = input.new_empty(n, taps, c)
        out = input.new_empty(n, c, oh.value, ow.value)
        strides = (ctypes.c_int64 * 4)(taps * c, 1, kernel_size * c, c)
        with torch.cuda.device(input.device):
            st = _lib.stream_ptr(input)
            _lib.check(L.dk_global_kernels_forward(
                desc, _lib.ptr(input), _lib.ptr(fc_weight), _lib.ptr(fc_bias), _lib.ptr(weight), _lib.ptr(pooled),
                _lib.ptr(coord[0]), _lib.ptr(coord[1]), _lib.ptr(kernels), st), "global_deform_conv kernels")
            _lib.check(L.dk_image_depthwise_forward(desc, _lib.ptr(input), _lib.ptr(kernels), strides, _lib.ptr(out), st),
                       "global_deform_conv forward")
        ctx.save_for_backward(input, weight, fc_weight, pooled, coord, kernels)
        ctx.desc, ctx.strides = desc, strides
        return out

    @staticmethod
    @once_differentiable  # the kernels are not differentiable a second time: asking for it raises
    def backward(ctx, grad_output):
        input, weight, fc_weight, pooled, coord, kernels = ctx.saved_tensors
        grad_output = grad_output.contiguous()
        need_input, need_weight, need_fc_w, need_fc_b = ctx.needs_input_grad[:4]
        L, p, desc = _lib.lib(), _lib.ptr, ctx.desc
        gx = gw = gfw = gfb = None
        with torch.cuda.device(input.device):
            st = _lib.stream_ptr(input)
            gk = torch.empty_like(kernels)
            _lib.check(L.dk_image_depthwise_backward_weight(desc, p(grad_output), p(input), p(gk), ctx.strides, st),
                       "global_deform_conv grad kernels")
            gpool = torch.empty(pooled.shape, dtype=torch.float32, device=input.device) if need_input else None
            gw = torch.empty_like(weight) if need_weight else None
            gfw = torch.empty_like(fc_weight) if need_fc_w else None
            gfb = fc_weight.new_empty(fc_weight.size(0)) if need_fc_b else None
            ws, nbytes = _lib.workspace(L.dk_global_kernels_backward_workspace(desc), input.device)
            _lib.check(L.dk_global_kernels_backward(
                desc, p(gk), p(pooled), p(coord[0]), p(coord[1]), p(weight), p(fc_weight), p(gw), p(gfw), p(gfb), p(gpool),
                p(ws), nbytes, st), "global_deform_conv grad parameters")
            if need_input:
                gx = torch.empty_like(input)
                _lib.check(L.dk_image_depthwise_backward_data_add(desc, p(grad_output), p(kernels), ctx.strides, p(gpool),
                                                                  p(gx), st), "global_deform_conv grad input")
        return gx, gw, gfw, gfb, None, None, None, None


def global_deform_conv(input, weight, fc_weight, fc_bias, kernel_size, stride=1, padding=0, dilation=1):
    return GlobalDeformConvFunction.apply(input, weight, fc_weight, fc_bias, kernel_size, _pair(stride), _pair(padding),
                                          _pair(dilation))
