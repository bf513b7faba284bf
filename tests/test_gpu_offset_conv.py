"""The offset branch's 3x3 convolution (the library's kernels for LocalDeformKernel2d's
rotation_conv) against the float64 convolution computed on the CPU: every pass within 1e-5 of it
(relative to its largest magnitude) for float32 tensors -- as bfloat16 pairs on the 16-bit matrix
instructions, and with that switched off as the fp32 matrix-instruction forward -- within the
results' own rounding for 16-bit tensors, and the module with the kernels switched on and off."""
import contextlib

import pytest
import torch
import torch.nn.functional as F

from _cases import rel_err

pytestmark = pytest.mark.gpu


def reference(x, w, b, gout=None, stride=1):
    """float64 convolution on the CPU of the tensors' values: out (and gx, gw, gb for a gout, which may be a
    function of the output's shape)."""
    xd, wd, bd = [t.detach().cpu().double().requires_grad_() for t in (x, w, b)]
    out = F.conv2d(xd, wd, bd, stride=stride, padding=1)
    if gout is None:
        return out.detach()
    out.backward(gout.detach().cpu().double())
    return out.detach(), xd.grad, wd.grad, bd.grad


def switches(pairs):
    from deformable_kernels.ops.deform_kernel import _lib
    return contextlib.nullcontext() if pairs else _lib.test_switches("DK_NO_OFFSET_PAIRS")


@pytest.mark.parametrize("shape", [
    (2, 16, 5, 7, 18),      # N, C, H, W, out channels: one partial tile
    (3, 32, 14, 14, 18),
    (2, 48, 28, 28, 18),    # tile rows 8: the last tile has 4 rows
    (2, 144, 56, 56, 18),   # the headline layer's offset branch
    (1, 32, 9, 112, 18),    # two 64-column segments per staged row, tile rows 4
    (2, 32, 56, 56, 16),    # no outputs beyond the matrix-core tile
    (2, 32, 20, 56, 8),     # fewer than 16 outputs
    (1, 16, 13, 28, 20),    # four outputs on the vector path
])
@pytest.mark.parametrize("pairs", [True, False])
def test_forward_matches_float64_convolution(shape, pairs):
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    N, C, H, W, O = shape
    g = torch.Generator().manual_seed(31)
    dev = torch.device("cuda:0")
    x = torch.randn(N, C, H, W, generator=g).to(dev)
    w = (torch.randn(O, C, 3, 3, generator=g) * 0.05).to(dev)
    b = torch.randn(O, generator=g).to(dev)
    with switches(pairs):
        assert offset_conv_supported(x, w, b, 1, 1, 1)
        got = offset_conv(x, w, b, force=True)
    want = reference(x, w, b)
    assert got.shape == want.shape and got.dtype == torch.float32
    assert rel_err(got.cpu(), want) < 1e-5


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float16, 2e-3), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("shape", [
    (2, 80, 5, 7, 18),      # a pixel per staged item, three chunks of 16-bit channels, the last half full
    (2, 48, 17, 14, 18),    # a plane lower than the tile
    (1, 96, 33, 28, 18),    # a third tile of one row
    (2, 48, 9, 56, 16),     # one block of outputs
    (1, 144, 5, 112, 18),   # five chunks, split between workgroups
])
@pytest.mark.parametrize("offset", [0, 1])  # 1: tensors that start between two aligned pairs of elements
def test_staged_pairs_of_pixels_and_tensors_off_their_alignment(shape, dtype, tol, offset):
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    N, C, H, W, O = shape
    g = torch.Generator().manual_seed(37)
    dev = torch.device("cuda:0")

    def tensor(*size, std=1.0):
        n = torch.Size(size).numel()
        return (torch.randn(n + offset, generator=g) * std).to(dtype).to(dev)[offset:].view(size)

    x, w, b, gout = tensor(N, C, H, W), tensor(O, C, 3, 3, std=0.05), tensor(O), tensor(N, O, H, W)
    x.requires_grad_()
    out = offset_conv(x, w, b, force=True)
    gx, = torch.autograd.grad(out, x, gout)
    want, want_gx, _, _ = reference(x, w, b, gout)
    assert rel_err(out.detach().float().cpu(), want) < tol
    assert rel_err(gx.float().cpu(), want_gx) < tol


@pytest.mark.parametrize("shape", [
    (2, 16, 5, 7, 18), (3, 32, 14, 14, 18), (2, 48, 28, 28, 18), (2, 144, 56, 56, 18), (1, 32, 9, 112, 18),
    (2, 32, 56, 56, 16), (1, 16, 13, 28, 20), (40, 32, 56, 56, 18),   # the last: several items per workgroup
])
@pytest.mark.parametrize("pairs", [True, False])   # False: the fp32 matrix-instruction weight gradient as well
def test_gradients_match_float64(shape, pairs):
    """float32 tensors: input gradient on the bfloat16-pair kernel (the framework's with the pairs off), weight
    gradient on the fp32 matrix instructions, bias gradient by the library's reduction."""
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    N, C, H, W, O = shape
    g = torch.Generator().manual_seed(33)
    dev = torch.device("cuda:0")
    x = torch.randn(N, C, H, W, generator=g).to(dev).requires_grad_()
    w = (torch.randn(O, C, 3, 3, generator=g) * 0.05).to(dev).requires_grad_()
    b = torch.randn(O, generator=g).to(dev).requires_grad_()
    gout = torch.randn(N, O, H, W, generator=g).to(dev)
    with switches(pairs):
        offset_conv(x, w, b, force=True).backward(gout)
    _, gx, gw, gb = reference(x, w, b, gout)
    assert rel_err(w.grad.cpu(), gw) < 1e-5
    assert rel_err(b.grad.cpu(), gb) < 1e-5
    assert rel_err(x.grad.cpu(), gx) < 1e-5


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-3), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("shape", [(2, 16, 5, 7, 18), (3, 32, 14, 14, 18), (2, 144, 56, 56, 18), (1, 32, 9, 112, 18),
                                   (2, 32, 56, 56, 16), (40, 32, 56, 56, 18), (64, 960, 7, 7, 18),
                                   (3, 192, 28, 28, 18), (2, 48, 13, 28, 18), (1, 16, 3, 56, 18), (2, 80, 21, 112, 20)])
def test_sixteen_bit_tensors_match_float64_on_the_rounded_inputs(shape, dtype, tol):
    """float16 / bfloat16 tensors: fp32 sums of exact products everywhere, so the error against the float64
    convolution of the rounded inputs is the results' own rounding.  Planes 28, 56 and 112 wide take the forward
    and the input gradient on the 16-bit matrix-instruction kernel (whole and partial row tiles, channel counts
    that leave half a chunk of 32, 16 / 18 / 20 outputs), the others the fp32-arithmetic forward and the
    library's input gradient; weight and bias gradient have fp32 partial sums."""
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    N, C, H, W, O = shape
    g = torch.Generator().manual_seed(37)
    dev = torch.device("cuda:0")
    x = torch.randn(N, C, H, W, generator=g).to(dtype).to(dev).requires_grad_()
    w = (torch.randn(O, C, 3, 3, generator=g) * 0.05).to(dtype).to(dev).requires_grad_()
    b = torch.randn(O, generator=g).to(dtype).to(dev).requires_grad_()
    gout = torch.randn(N, O, H, W, generator=g).to(dtype).to(dev)
    assert offset_conv_supported(x, w, b, 1, 1, 1)
    out = offset_conv(x, w, b, force=True)
    assert out.dtype == dtype
    out.backward(gout)
    want, gx, gw, gb = reference(x, w, b, gout)
    assert rel_err(out.detach().double().cpu(), want) < tol
    assert w.grad.dtype == dtype and b.grad.dtype == dtype
    assert rel_err(w.grad.double().cpu(), gw) < tol
    assert rel_err(b.grad.double().cpu(), gb) < tol
    assert x.grad.dtype == dtype
    assert rel_err(x.grad.double().cpu(), gx) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float16, 2e-3), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("shape", [(2, 96, 112, 112, 18), (3, 144, 56, 56, 18), (2, 192, 28, 28, 18), (5, 576, 14, 14, 18),
                                   (2, 32, 9, 56, 18), (1, 16, 1, 14, 16), (2, 48, 30, 28, 20), (2, 32, 17, 112, 7)])
def test_stride_2_forward_and_input_gradient(shape, dtype, tol):
    """The down-sampling layers' convolution (stride 2, padding 1): forward and input gradient on the 16-bit matrix
    instructions -- float16 / bfloat16 elements as they are, float32 ones as bfloat16 pairs (two chunks of output
    gradient channels in the input gradient) -- over whole, partial and single-row tiles, odd heights, half
    chunks of channels, planes lower than a tile, chunk splits, one to three blocks of 16 channels; the weight
    gradient on the framework's routine, the bias gradient on the library's."""
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    N, C, H, W, O = shape
    g = torch.Generator().manual_seed(43)
    dev = torch.device("cuda:0")
    x = torch.randn(N, C, H, W, generator=g).to(dtype).to(dev).requires_grad_()
    w = (torch.randn(O, C, 3, 3, generator=g) * 0.05).to(dtype).to(dev).requires_grad_()
    b = torch.randn(O, generator=g).to(dtype).to(dev).requires_grad_()
    assert offset_conv_supported(x, w, b, 2, 1, 1)
    if dtype == torch.float32:
        with switches(False):
            assert not offset_conv_supported(x, w, b, 2, 1, 1)
    out = offset_conv(x, w, b, stride=2, force=True)
    gout = torch.randn(out.shape, generator=g).to(dtype).to(dev)
    want, gx, gw, gb = reference(x, w, b, gout, stride=2)
    assert out.shape == want.shape and out.dtype == dtype
    assert rel_err(out.detach().double().cpu(), want) < tol
    out.backward(gout)
    assert rel_err(x.grad.double().cpu(), gx) < tol
    assert rel_err(w.grad.double().cpu(), gw) < tol
    assert rel_err(b.grad.double().cpu(), gb) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("wgrad16", [True, False])
def test_fewer_than_15_outputs(dtype, tol, wgrad16):
    """Seven outputs: every pass has a kernel on the 16-bit matrix instructions; with that weight gradient switched
    off the fp32 matrix-instruction one, which covers 15 and more outputs, answers its workspace query with 0 and
    the weight gradient comes from the framework's routine."""
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    g = torch.Generator().manual_seed(41)
    dev = torch.device("cuda:0")
    x = torch.randn(2, 32, 9, 56, generator=g).to(dtype).to(dev).requires_grad_()
    w = (torch.randn(7, 32, 3, 3, generator=g) * 0.05).to(dtype).to(dev).requires_grad_()
    b = torch.randn(7, generator=g).to(dtype).to(dev).requires_grad_()
    gout = torch.randn(2, 7, 9, 56, generator=g).to(dtype).to(dev)
    from deformable_kernels.ops.deform_kernel import _lib
    with contextlib.nullcontext() if wgrad16 else _lib.test_switches("DK_NO_OFFSET_WGRAD16"):
        assert offset_conv_supported(x, w, b, 1, 1, 1)
        assert (_lib.lib().dk_offset_conv_backward_weight_workspace(
            _lib.OffsetConvDesc(2, 32, 7, 9, 56, _lib.dtype_tag(x), 1)) > 0) == wgrad16
        out = offset_conv(x, w, b, force=True)
        out.backward(gout)
    want, gx, gw, gb = reference(x, w, b, gout)
    for got, ref in ((out.detach(), want), (x.grad, gx), (w.grad, gw), (b.grad, gb)):
        assert got.dtype == dtype and rel_err(got.double().cpu(), ref) < tol


def test_unsupported_calls_go_to_the_library_convolution():
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    dev = torch.device("cuda:0")
    x = torch.randn(2, 24, 10, 10, device=dev)   # 24 channels: not a multiple of 16; width 10
    w = torch.randn(18, 24, 3, 3, device=dev)
    assert not offset_conv_supported(x, w, None, 1, 1, 1)
    assert torch.equal(offset_conv(x, w, None), F.conv2d(x, w, None, 1, 1, 1))
    x2 = torch.randn(2, 32, 56, 56, device=dev)
    w2 = torch.randn(18, 32, 3, 3, device=dev)
    with switches(False):
        assert not offset_conv_supported(x2, w2, None, 2, 1, 1)      # stride 2, float32, without the pair kernels
    assert not offset_conv_supported(x2[:, :, :, :20].contiguous(), w2, None, 2, 1, 1)   # stride 2, 20 columns
    assert not offset_conv_supported(x2.double(), w2.double(), None, 1, 1, 1)   # float64
    assert not offset_conv_supported(x2.half(), w2, None, 1, 1, 1)              # mixed dtypes
    with switches(False):
        assert torch.equal(offset_conv(x2, w2, None, stride=2), F.conv2d(x2, w2, None, 2, 1, 1))
    assert torch.equal(offset_conv(x2.double(), w2.double(), None), F.conv2d(x2.double(), w2.double(), None, 1, 1, 1))


@pytest.mark.parametrize("conv", [(2, 1, 1), (1, 0, 1), (1, 2, 2), (2, 1, 1, 24)])
def test_other_convolutions_keep_the_library_kernels_but_not_its_bias_gradient(conv):
    # stride 2 / no padding / dilation 2 / 24 channels: the forward is F.conv2d's, the gradients match autograd's
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    stride, padding, dilation = conv[:3]
    C = conv[3] if len(conv) > 3 else 32
    g = torch.Generator().manual_seed(34)
    dev = torch.device("cuda:0")
    x = torch.randn(3, C, 20, 22, generator=g).to(dev).requires_grad_()
    w = (torch.randn(18, C, 3, 3, generator=g) * 0.05).to(dev).requires_grad_()
    b = torch.randn(18, generator=g).to(dev).requires_grad_()
    out = offset_conv(x, w, b, stride, padding, dilation)
    x2, w2, b2 = [t.detach().clone().requires_grad_() for t in (x, w, b)]
    ref = F.conv2d(x2, w2, b2, stride, padding, dilation)
    assert torch.equal(out, ref)
    gout = torch.randn(ref.shape, generator=g).to(dev)
    out.backward(gout)
    ref.backward(gout)
    assert rel_err(x.grad.cpu(), x2.grad.cpu()) < 1e-6
    assert rel_err(w.grad.cpu(), w2.grad.cpu()) < 1e-6
    assert rel_err(b.grad.cpu(), gout.double().sum((0, 2, 3)).float().cpu()) < 1e-5


def test_gradients_and_module_switch():
    from deformable_kernels.modules import LocalDeformKernel2d
    torch.manual_seed(32)
    dev = torch.device("cuda:0")
    C = 16
    m = LocalDeformKernel2d((4, 4), C, C, 3, 1, 1, 1, C, 1, False, 'scope').to(dev)
    torch.nn.init.normal_(m.rotation_conv.weight, std=0.1)
    x = torch.randn(28, C, 56, 56, device=dev)    # 28 images x 7 row tiles: the native kernel is chosen
    gout = torch.randn(28, C, 56, 56, device=dev)
    results = []
    for native, pairs in ((False, True), (True, True), (True, False)):
        m.native_offset_conv = native
        m.zero_grad()
        xi = x.clone().requires_grad_()
        with switches(pairs):
            out = m(xi)
            out.backward(gout)
        results.append([t.detach().cpu().clone() for t in (
            out, xi.grad, m.inner_conv.weight.grad, m.rotation_conv.weight.grad, m.rotation_conv.bias.grad)])
    # The branch's float32 kernels multiply bfloat16 pairs (3.5e-6 of the rotations' scale) and the operator's
    # output moves with its rotations: 1.7e-5 of the output's scale was measured here.  Its rotation gradient is
    # piecewise constant in the rotation (the slope of the bilinear patch): a rotation within that distance of a
    # cell border lands in the neighbouring cell and moves one element of the rotation gradient -- and the 144
    # input-gradient elements under it -- by a finite amount.  About ten of the 1.6 M coordinates do, so the
    # gradients are compared in the root mean square and by the share of elements that moved at all; with the
    # pairs switched off (5e-7) none flips and the element-wise bound holds.
    assert rel_err(results[1][0], results[0][0]) < 5e-5
    for got, ref in zip(results[1][1:], results[0][1:]):
        diff = (got - ref).abs()
        assert float(diff.pow(2).mean().sqrt() / ref.pow(2).mean().sqrt()) < 1e-2   # (2.2e-3 measured)
        if got.numel() > 100000:   # the input gradient: few elements move at all (the others are sums over pixels)
            assert float((diff > 1e-4 * ref.abs().max()).float().mean()) < 5e-3
    assert rel_err(results[2][0], results[0][0]) < 1e-5
    for got, ref in zip(results[2][1:], results[0][1:]):
        assert rel_err(got, ref) < 1e-4


@pytest.mark.parametrize("case", [
    # one image, three groups of six outputs; fewer channels than waves; a partial last group of four channels
    (1, 192, 28, 28, 18, 1, "float32"), (1, 16, 7, 7, 18, 1, "float32"), (2, 80, 14, 14, 18, 1, "bfloat16"),
    # 128 tiles of 64 pixels and more: all outputs in one workgroup; pixels no multiple of 64
    (2, 32, 112, 112, 18, 1, "float32"), (3, 48, 53, 56, 18, 1, "float16"),
    # the weight gradient's form for 256 channels and more, one row of pixels
    (5, 256, 14, 14, 18, 1, "float32"), (1, 272, 1, 7, 7, 1, "float16"),
    # stride 2: odd heights, fewer outputs than a workgroup's
    (2, 32, 5, 14, 18, 2, "float32"), (15, 192, 28, 28, 18, 2, "bfloat16"), (1, 16, 56, 56, 1, 2, "float32"),
])
def test_few_images_run_on_the_vector_unit_kernels(case):
    """Forward, input and weight gradient of batches too small for the matrix-instruction kernels against the float64
    convolution: every sum is float32 over at most 9 * 272 (forward) or 25088 / 64 pixel groups (weight gradient) terms in
    parts of at most 162, so 2e-6 of the largest element; 16-bit results are rounded once (2^-11, 2^-8)."""
    from deformable_kernels.ops.deform_kernel import _lib
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    N, C, H, W, O, stride, dtype_name = case
    dtype = getattr(torch, dtype_name)
    tol = {"float32": 2e-6, "float16": 5e-4 + 2e-6, "bfloat16": 4e-3 + 2e-6}[dtype_name]
    desc = _lib.OffsetConvDesc(N, C, O, H, W, {"float32": 0, "float16": 1, "bfloat16": 2}[dtype_name], stride)
    assert _lib.lib().dk_offset_conv_direct_worthwhile(desc) == 1
    g = torch.Generator().manual_seed(71)
    dev = torch.device("cuda:0")
    x = torch.randn(N, C, H, W, generator=g).to(dtype).to(dev).requires_grad_()
    w = (torch.randn(O, C, 3, 3, generator=g) * 0.05).to(dtype).to(dev).requires_grad_()
    b = torch.randn(O, generator=g).to(dtype).to(dev).requires_grad_()
    out = offset_conv(x, w, b, stride)
    gout = torch.randn(out.shape, generator=g).to(dtype).to(dev)
    want, gx, gw, gb = reference(x, w, b, gout, stride=stride)
    out.backward(gout)
    assert rel_err(out.detach().double().cpu(), want) < tol, "forward"
    assert rel_err(x.grad.double().cpu(), gx) < tol, "input gradient"
    assert rel_err(w.grad.double().cpu(), gw) < tol, "weight gradient"


@pytest.mark.parametrize("forward, backward, case", [
    # either side of each line of the two rules: N, C, H, W, outputs, stride, dtype
    (1, 1, (1, 192, 28, 28, 18, 1, "float32")), (1, 1, (63, 608, 7, 7, 18, 1, "float32")),
    (0, 1, (3, 768, 7, 7, 18, 1, "float32")), (1, 1, (3, 736, 7, 7, 18, 1, "float32")), (1, 1, (1, 640, 14, 14, 18, 1, "bfloat16")),
    (0, 1, (1, 640, 14, 14, 18, 2, "bfloat16")), (1, 1, (1, 384, 14, 14, 18, 2, "float16")),
    (0, 1, (1, 320, 56, 56, 18, 2, "float32")), (1, 1, (1, 304, 56, 56, 18, 2, "float32")),
    (0, 1, (1, 960, 14, 14, 18, 1, "float16")), (1, 1, (2, 960, 14, 14, 18, 1, "float16")), (1, 1, (1, 960, 14, 14, 18, 1, "float32")),
    (0, 1, (11, 80, 28, 28, 18, 1, "float16")), (1, 1, (11, 64, 28, 28, 18, 1, "float16")), (1, 1, (11, 128, 28, 28, 18, 1, "float32")),
    (0, 1, (11, 144, 28, 28, 18, 1, "float32")), (1, 1, (11, 144, 28, 28, 18, 1, "bfloat16")),
    (1, 0, (17, 192, 28, 28, 18, 2, "float32")), (1, 1, (16, 192, 28, 28, 18, 2, "float32")),
])
def test_calls_that_take_the_vector_unit_kernels(forward, backward, case):
    """The rules, and the operator's own way through each combination of them against the float64 convolution.  The framework's
    kernels: 16-bit results up to two of whose roundings meet (2^-10, 2^-7); bounds of the vector-unit kernels as above with up to
    9 * 960 terms, and float32 sums of the framework of up to 1e-5."""
    from deformable_kernels.ops.deform_kernel import _lib
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    N, C, H, W, O, stride, dtype_name = case
    desc = _lib.OffsetConvDesc(N, C, O, H, W, {"float32": 0, "float16": 1, "bfloat16": 2}[dtype_name], stride)
    assert _lib.lib().dk_offset_conv_direct_worthwhile(desc) == forward
    assert _lib.lib().dk_offset_conv_direct_backward_worthwhile(desc) == backward
    if N * C * H * W > 1000000:
        return
    dtype = getattr(torch, dtype_name)
    tol = {"float32": 1e-5, "float16": 1e-3 + 1e-5, "bfloat16": 8e-3 + 1e-5}[dtype_name]
    g = torch.Generator().manual_seed(73)
    x, w, b = [t.to(dtype).cuda().requires_grad_() for t in (torch.randn(N, C, H, W, generator=g), torch.randn(O, C, 3, 3, generator=g) * 0.05,
                                                             torch.randn(O, generator=g))]
    out = offset_conv(x, w, b, stride)
    gout = torch.randn(out.shape, generator=g).to(dtype).cuda()
    want = reference(x, w, b, gout, stride=stride)
    out.backward(gout)
    for name, got, ref in zip(("forward", "input", "weight", "bias"), (out.detach(), x.grad, w.grad, b.grad), want):
        assert rel_err(got.double().cpu(), ref) < tol, name


@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("case", [
    (1, 10, 1, 1, 5, 1),      # one pixel: eight of nine taps in the padding; fewer channels than waves
    (2, 7, 9, 13, 18, 1),     # a width no layer has
    (3, 33, 13, 5, 1, 2),     # one output, odd sides at stride 2
    (1, 300, 2, 65, 17, 1),   # the weight gradient's form for 256 channels and more; a row wider than a wave
    (70, 3, 11, 13, 4, 1),    # more than 128 tiles of pixels
    (2, 20, 3, 4, 18, 2),
])
def test_vector_unit_entry_points_on_sizes_that_the_operator_leaves_to_the_framework(case, dtype_name):
    """The three C calls take any size: float32 sums of at most 9 * 300 terms (2e-6 of the largest element), one rounding of a 16-bit
    result (2^-11, 2^-8)."""
    from deformable_kernels.ops.deform_kernel import _lib
    N, C, H, W, O, stride = case
    dtype = getattr(torch, dtype_name)
    tol = {"float32": 2e-6, "float16": 5e-4 + 2e-6, "bfloat16": 4e-3 + 2e-6}[dtype_name]
    g = torch.Generator().manual_seed(79)
    x, w, b, gout = [t.to(dtype).cuda() for t in (torch.randn(N, C, H, W, generator=g), torch.randn(O, C, 3, 3, generator=g) * 0.05,
                                                 torch.randn(O, generator=g), torch.randn(N, O, (H - 1) // stride + 1, (W - 1) // stride + 1, generator=g))]
    out, gx, gw = torch.full_like(gout, float("nan")), torch.full_like(x, float("nan")), torch.full_like(w, float("nan"))
    L, P = _lib.lib(), _lib.ptr
    desc = _lib.OffsetConvDesc(N, C, O, H, W, {"float32": 0, "float16": 1, "bfloat16": 2}[dtype_name], stride)
    st = _lib.stream_ptr(x)
    _lib.check(L.dk_offset_conv_direct_forward(desc, P(x), P(w), P(b), P(out), st), "forward")
    _lib.check(L.dk_offset_conv_direct_backward_input(desc, P(gout), P(w), P(gx), st), "input gradient")
    _lib.check(L.dk_offset_conv_direct_backward_weight(desc, P(gout), P(x), P(gw), st), "weight gradient")
    want = reference(x, w, b, gout, stride=stride)
    for name, got, ref in zip(("forward", "input", "weight"), (out, gx, gw), want):
        assert rel_err(got.double().cpu(), ref) < tol, name


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-3), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("shape", [
    (2, 1, 5, 7, 1),         # N, C, H, W, stride: one channel
    (3, 17, 14, 14, 1),      # a chunk of sixteen and one of one
    (2, 33, 28, 28, 1),      # two of the forward's chunks, the second of one channel
    (2, 61, 9, 56, 1),
    (1, 41, 6, 112, 1),
    (2, 15, 13, 28, 2),
    (2, 50, 14, 14, 2),
    (1, 37, 10, 112, 2),
])
def test_any_number_of_channels_in_16_bits(shape, dtype, tol):
    """Forward and both gradients on the 16-bit matrix instructions: the last chunk's missing channels read as zeros, whatever lies
    behind the tensor."""
    from deformable_kernels.ops.deform_kernel.functions import offset_conv, offset_conv_supported
    N, C, H, W, s = shape
    g = torch.Generator().manual_seed(41)
    behind = torch.full((N * C * H * W + 64 * H * W,), float("nan"), device="cuda:0", dtype=dtype)
    x = behind[:N * C * H * W].view(N, C, H, W).copy_(torch.randn(N, C, H, W, generator=g))
    w = (torch.randn(18, C, 3, 3, generator=g) / (9 * C) ** 0.5).to(dtype).cuda()
    b = torch.randn(18, generator=g).to(dtype).cuda()
    leaves = [t.requires_grad_() for t in (x, w, b)]
    assert offset_conv_supported(x, w, b, s, 1, 1)
    out = offset_conv(x, w, b, s, force=True)
    gout = torch.randn(out.shape, generator=g).to(dtype).cuda()
    got = (out.detach(),) + torch.autograd.grad(out, leaves, gout)
    for a, want in zip(got, reference(x, w, b, gout, s)):
        assert a.dtype == dtype and rel_err(a.float().cpu(), want) < tol


@pytest.mark.parametrize("shape,dtype", [
    ((35, 15, 17, 19, 1), torch.float16), ((2, 300, 33, 35, 2), torch.float16), ((10, 60, 10, 11, 1), torch.bfloat16),
])
def test_gradients_of_few_images_on_any_plane(shape, dtype):
    from deformable_kernels.ops.deform_kernel.functions import offset_conv
    N, C, H, W, s = shape
    g = torch.Generator().manual_seed(42)
    leaves = [(torch.randn(N, C, H, W, generator=g)).to(dtype).cuda().requires_grad_(),
              (torch.randn(18, C, 3, 3, generator=g) / (9 * C) ** 0.5).to(dtype).cuda().requires_grad_(),
              torch.randn(18, generator=g).to(dtype).cuda().requires_grad_()]
    out = offset_conv(*leaves, s)
    gout = torch.randn(out.shape, generator=g).to(dtype).cuda()
    got = torch.autograd.grad(out, leaves, gout)
    tol = 2e-3 if dtype == torch.float16 else 1e-2
    assert torch.equal(out, F.conv2d(*leaves, s, 1))  # the offsets are the framework's
    for a, want in zip(got, reference(*leaves, gout, s)[1:]):
        assert rel_err(a.float().cpu(), want) < tol
