"""The work that a user of this library has it do, as measurable cases.

``listed()`` are the named cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` makes what a
user's program holds before the call, ``run`` is one pass through the public entry points: the autograd Functions
``sample_depthwise``, ``deform_sample_depthwise`` and ``nd_linear_sample``, and the layers ``DeformKernel2d``,
``DeformKernelConv2d`` and ``GlobalDeformKernel2d``.  A training pass is the forward call, then the gradients of
everything that is trained for a given upstream gradient; an inference pass is the forward call without a graph.

Kinds of case
  local        sample_depthwise on given kernel-space offsets (``x, rotation, weight``)
  deform       deform_sample_depthwise on given image-space and kernel-space offsets
  layer        DeformKernel2d: the 3 x 3 offset branch and the operator, as a network calls it
  conv_layer   DeformKernelConv2d: the same with image-space offsets (no kernel-space ones)
  global       GlobalDeformKernel2d: one set of kernel-space offsets per image from the pooled input
  nd           nd_linear_sample on a 1-d, 2-d or 3-d grid
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "deformable-kernels_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

from deformable_kernels.modules import DeformKernel2d, DeformKernelConv2d, GlobalDeformKernel2d
from deformable_kernels.ops.deform_kernel.functions import (
    deform_sample_depthwise, nd_linear_sample, sample_depthwise)

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}
_TAPS = 9  # every convolution here has 3 x 3 taps and padding 1, as the networks' depthwise layers do


def _conv(name, kind, n, c, h, w, dtype, stride=1, scope=4, groups=1, layout="nchw", train=True):
    case = dict(kind=kind, n=n, c=c, h=h, w=w, dtype=dtype, stride=stride, scope=scope, groups=groups,
                layout=layout, train=train)
    return dict(name=name, **case) if name else case


def _nd(name, c, shape, points, dtype):
    shape = list(shape) + [1] * (3 - len(shape))  # trailing extents of 1: dimensions the grid does not have
    case = dict(kind="nd", c=c, s0=shape[0], s1=shape[1], s2=shape[2], points=points, dtype=dtype, train=True)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # a small layer in a unit-sized batch: what a first experiment runs, and all launch latency
        _conv("local_small_fp32", "local", 2, 32, 28, 28, "fp32"),
        # one image through one layer of a deployed network
        _conv("layer_one_image_infer_fp32", "layer", 1, 192, 28, 28, "fp32", train=False),
        # the large middle stage of MobileNetV2-DK at batch 64
        _conv("local_56_fp32", "local", 64, 144, 56, 56, "fp32"),
        # its late stage in a 16-bit training run at batch 128: small planes, many channels
        _conv("local_14_bf16", "local", 128, 576, 14, 14, "bf16"),
        # planes no network table has: odd sizes, a channel count that is no multiple of 16, two rotation groups,
        # a larger scope -- segmentation crops and other users' own layers
        _conv("local_odd_fp32", "local", 12, 90, 75, 101, "fp32", scope=5, groups=2),
        # the first down-sampling layer of a network that keeps its tensors channels-last, 16-bit
        _conv("local_112_stride2_nhwc_bf16", "local", 64, 96, 112, 112, "bf16", stride=2, layout="nhwc"),
        # a layer with its offset branch, as a 16-bit training run of the network meets it 17 times a step
        _conv("layer_28_train_bf16", "layer", 128, 192, 28, 28, "bf16"),
        # image-space and kernel-space offsets together on a down-sampling layer with many channels
        _conv("deform_28_stride2_fp32", "deform", 64, 512, 28, 28, "fp32", stride=2),
        # ... and on the large middle stage: the costliest pass of the library
        _conv("deform_56_fp32", "deform", 64, 144, 56, 56, "fp32"),
        # the image-space layer with its offset branch in a 16-bit training run
        _conv("conv_layer_28_train_fp16", "conv_layer", 64, 192, 28, 28, "fp16"),
        # the per-image layer, 16-bit
        _conv("global_28_train_fp16", "global", 128, 256, 28, 28, "fp16", scope=5),
        # the sampler by itself: a million points in a volume of feature vectors
        _nd("nd_volume_fp32", 64, (32, 32, 32), 1 << 20, "fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# kind: (most elements of the input, widest plane, scopes); a drawn input stays below the listed ones' cost
_RANGES = {
    "local": (12_000_000, 128, (3, 4, 4, 5, 7)),
    "layer": (12_000_000, 112, (4,)),
    "deform": (6_000_000, 112, (3, 4, 4, 5)),
    "conv_layer": (6_000_000, 112, (4,)),
    "global": (25_000_000, 112, (4, 5)),
}


def draw(rng):
    kind = rng.choice(("local", "local", "local", "layer", "deform", "conv_layer", "global", "nd"))
    dtype = rng.choice(("fp32", "fp16", "bf16"))
    if kind == "nd":
        dims = rng.choice((1, 2, 2, 3, 3))
        c = _log_int(rng, 3, 256)
        shape = [_log_int(rng, 4, (4096, 96, 40)[dims - 1]) for _ in range(dims)]
        points = min(_log_int(rng, 500, 1 << 20), (1 << 26) // c)
        return _nd(None, c, shape, points, dtype)
    most, widest, scopes = _RANGES[kind]
    if rng.random() < 0.5:  # a network's own plane, else any
        h = w = rng.choice([s for s in (7, 14, 28, 56, 112) if s <= widest])
    else:
        h, w = _log_int(rng, 7, widest), _log_int(rng, 7, widest)
    c = 16 * _log_int(rng, 1, 60) if rng.random() < 0.6 else _log_int(rng, 10, 600)
    groups = 1
    if kind in ("local", "deform") and rng.random() < 0.2:
        groups, c = 2, c + c % 2
    n = max(1, min(_log_int(rng, 1, 128), most // (c * h * w)))
    stride = rng.choice((1, 1, 2)) if min(h, w) >= 14 else 1
    layout = "nhwc" if kind in ("local", "layer") and rng.random() < 0.2 else "nchw"
    return _conv(None, kind, n, c, h, w, dtype, stride, rng.choice(scopes), groups, layout, rng.random() < 0.75)


def _out_plane(case):
    return (case["h"] - 1) // case["stride"] + 1, (case["w"] - 1) // case["stride"] + 1


class _Inputs:
    """Tensors on the GPU from one seed."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = _DTYPES[case["dtype"]]

    def normal(self, shape, std=1.0, channels_last=False):
        t = (torch.randn(shape, generator=self.gen, device="cuda") * std).to(self.dtype)
        return t.contiguous(memory_format=torch.channels_last) if channels_last else t

    def uniform(self, shape, lo, hi):
        return (torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo).to(self.dtype)

    def fill(self, parameter, std):
        parameter.data = self.normal(parameter.shape, std)


def _layer(case, rand):
    """The layer as a trained network holds it: an offset branch that predicts offsets of the usual size."""
    c, scope = case["c"], (case["scope"], case["scope"])
    kind = {"layer": DeformKernel2d, "conv_layer": DeformKernelConv2d, "global": GlobalDeformKernel2d}[case["kind"]]
    module = kind(scope, c, c, kernel_size=3, stride=case["stride"], padding=1, groups=c).to(rand.dtype).cuda()
    if case["kind"] == "global":
        # the inputs' channel means are ~ N(0, 1 / (h * w)); the pooled branch makes offsets ~ N(0, 0.5) of them
        rand.fill(module.fc.weight, 0.5 * math.sqrt(case["h"] * case["w"] / c))
        rand.fill(module.fc.bias, 0.1)
        rand.fill(module.weight, math.sqrt(2.0) / 3.0)
    else:
        branch = module.rotation_conv if case["kind"] == "layer" else module.offset_conv
        rand.fill(branch.weight, (0.5 if case["kind"] == "layer" else 2.0) / math.sqrt(9 * c))
        rand.fill(branch.bias, 0.3)
        rand.fill(module.inner_conv.weight, math.sqrt(2.0) / 3.0)
    return module.train(case["train"])


def prepare(case, seed):
    rand = _Inputs(case, seed)
    if case["kind"] == "nd":
        shape = [s for s in (case["s0"], case["s1"], case["s2"]) if s > 1]
        data = rand.normal([case["c"]] + shape)
        # all over the grid and up to a cell beyond it
        coord = torch.stack([rand.uniform([case["points"]], -1.0, float(s)) for s in shape], 1)
        grad = rand.normal((case["points"], case["c"]))
        return _state(case, nd_linear_sample, [data, coord], (), [data, coord], grad)
    n, c, h, w, groups = (case[k] for k in ("n", "c", "h", "w", "groups"))
    oh, ow = _out_plane(case)
    last = case["layout"] == "nhwc"
    x = rand.normal((n, c, h, w), channels_last=last)
    grad = rand.normal((n, c, oh, ow), channels_last=last)
    if case["kind"] in ("local", "deform"):
        weight = rand.normal((c, 1, case["scope"], case["scope"]), math.sqrt(2.0) / 3.0)
        rotation = rand.normal((n, groups * 2 * _TAPS, oh, ow), 0.7, channels_last=last)
        options = ((3, 3), (case["stride"],) * 2, (1, 1), (1, 1), groups)
        if case["kind"] == "local":
            call, args = sample_depthwise, [x, rotation, weight]
        else:
            call, args = deform_sample_depthwise, [x, rand.normal((n, 2 * _TAPS, oh, ow), 2.0), rotation, weight]
        leaves = args
    else:
        call, args, options = _layer(case, rand), [x], ()
        leaves = [x] + list(call.parameters())
    return _state(case, call, args, options, leaves, grad)


def _state(case, call, args, options, leaves, grad):
    for t in leaves:
        t.requires_grad_(case["train"])
    return dict(call=call, args=args, options=options, leaves=leaves, grad=grad, train=case["train"])


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return state["call"](*state["args"], *state["options"])
    out = state["call"](*state["args"], *state["options"])
    return [out.detach()] + list(torch.autograd.grad(out, state["leaves"], state["grad"]))


def work(case):
    """Every tensor of the pass read or written once, and the arithmetic of the definition."""
    size, train = _SIZE[case["dtype"]], case["train"]
    if case["kind"] == "nd":
        dims = sum(s > 1 for s in (case["s0"], case["s1"], case["s2"]))
        data, out = case["c"] * case["s0"] * case["s1"] * case["s2"], case["points"] * case["c"]
        corners = 2 ** dims
        # a corner's share of a channel: one multiply-add forward, one for the data gradient, one per
        # dimension (by halves: the differences are shared) for the coordinates' gradient
        return {"bytes": size * (2 * data + 2 * out + 2 * case["points"] * dims), "flops": 2 * out * corners * 3}
    n, c, h, w = (case[k] for k in ("n", "c", "h", "w"))
    oh, ow = _out_plane(case)
    x, out, weight = n * c * h * w, n * c * oh * ow, c * case["scope"] ** 2
    passes = 2 if train else 1
    if case["kind"] == "global":
        branch = c * 2 * _TAPS + 2 * _TAPS
        # one multiply-add per tap and output forward, for the input's and for the kernels' gradient
        return {"bytes": size * passes * (x + out + weight + branch), "flops": 2 * _TAPS * out * (3 if train else 1)}
    offsets = n * case["groups"] * 2 * _TAPS * oh * ow
    image = n * 2 * _TAPS * oh * ow
    deform = case["kind"] in ("deform", "conv_layer")
    # a bilinear read is four multiply-adds; each gradient's is as much again
    reads = (1 if case["kind"] != "deform" else 2) * 8
    flops = out * _TAPS * (reads + 2) * (4 if train else 1)
    if case["kind"] in ("layer", "conv_layer"):  # the offset branch's convolution; its offsets need not leave the chip
        branch = 2 * _TAPS * _TAPS * c
        flops += 2 * branch * n * oh * ow * (3 if train else 1)
        return {"bytes": size * passes * (x + out + weight + branch), "flops": flops}
    return {"bytes": size * passes * (x + out + weight + offsets + (image if deform else 0)), "flops": flops}


# Measured, then times four: the operators and the sampler against themselves in float64 (float32: 4.4e-6 local,
# 2.3e-6 deform -- leaving out single samples whose float32 position falls on the other side of a grid line, where
# the slope jumps -- and 4e-7 nd; fp16 2.4e-3, bf16 3.6e-3, in the gradients that sum products of 16-bit operands);
# the layers against themselves with the offset branch's sums in another order.  A 16-bit offset that rounds the
# other way moves its sample by its last bit, and where it crosses a cell border the slope jumps: up to 3.2e-2 (bf16)
# and 2.9e-2 (fp16) of the gradients of `layer`, 1e-1 and 3e-2 of those of `conv_layer`, whose offsets are larger,
# 1.5e-3 and 4.3e-3 in float32.  The per-image layer has few offsets: rarely one moves.
_TOLERANCE = {
    "local": {"fp32": 2e-5, "fp16": 1e-2, "bf16": 1.5e-2},
    "deform": {"fp32": 2e-5, "fp16": 1e-2, "bf16": 1.5e-2},
    "layer": {"fp32": 6e-3, "fp16": 1.2e-1, "bf16": 1.3e-1},
    "conv_layer": {"fp32": 1.7e-2, "fp16": 1.2e-1, "bf16": 4e-1},
    "global": {"fp32": 3e-6, "fp16": 1e-2, "bf16": 3e-2},
    "nd": {"fp32": 2e-6, "fp16": 1e-3, "bf16": 8e-3},
}


def tolerance(case):
    return {"rel": _TOLERANCE[case["kind"]][case["dtype"]]}
