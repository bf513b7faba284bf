"""GPU parity of the deformable variant (kernel-space + image-space offsets):
forward, grad-input, grad-offset, grad-rotation, grad-filter against the CPU
oracle, through the Python Function and the C ABI.

Tolerances relative to the largest expected magnitude: fp32 forward 1e-5
against the fp32 oracle; the four gradients 1e-4 against the fp64 oracle
(grad-input is an atomic scatter, the others are reductions, so summation order
differs from the oracle's); fp64 1e-11; fp16 / bf16 1e-2 against the fp32
oracle on the rounded inputs."""
import numpy as np
import pytest
import torch

from _cases import mixed_err, clipped_rotation, make_deform, rel_err
from oracle import dk_oracle as orc

pytestmark = pytest.mark.gpu

# N, C, H, W, k, S, stride, pad, dil, groups, rot_std, off_std
CASES = [
    (2, 16, 14, 14, 3, (4, 4), 2, 1, 1, 1, 0.5, 2.0),     # benchmark configuration 4 geometry, small
    (2, 12, 13, 11, 3, (4, 4), 1, 1, 1, 1, 1.0, 2.0),
    (2, 12, 9, 10, 3, (4, 4), 1, 2, 2, 3, 0.7, 3.0),      # dilation, rotation groups
    (1, 8, 12, 12, 3, (3, 3), 1, 1, 1, 1, 0.0, 1.5),      # DeformConv2d: scope == kernel, zero rotation
    (2, 6, 8, 8, (2, 3), (4, 5), (1, 2), (0, 1), 1, 3, 0.7, 1.0),
    (1, 3, 6, 5, 1, (2, 2), 1, 0, 1, 1, 0.6, 3.0),
    (1, 20, 24, 24, 3, (4, 4), 1, 1, 1, 2, 0.7, 2.0),     # 576 output pixels: three pixel tiles, two groups
    (1, 6, 33, 60, 3, (5, 5), 1, 1, 1, 1, 1.0, 2.5),      # wide plane (16 staging passes), scope 5, > 1024 output pixels
    (2, 80, 10, 10, 3, (3, 3), 1, 1, 1, 1, 0.8, 1.0),     # many channels: several channel chunks per image
    (1, 8, 20, 18, 3, (4, 4), 2, 1, 1, 1, 0.5, 6.0),      # large offsets: many samples outside the image
    (2, 10, 40, 36, 3, (4, 4), 1, 1, 1, 2, 0.7, 2.0),     # 1440 output pixels: tiled grad input, 5 channels per group (partial chunk)
    (2, 27, 14, 14, 3, (4, 4), 2, 1, 1, 1, 0.5, 2.0),     # three chunks of 9 channels: the four-channel tuples end in a single channel
    (1, 9, 16, 17, 3, (5, 5), 1, 1, 1, 1, 1.0, 2.0),      # scope 5 on the channel-interleaved kernels
    (1, 9, 56, 56, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),      # 56 x 56: 512-thread channel-interleaved kernels, 7 tiles of 7 waves
    (1, 6, 64, 64, 3, (5, 5), 2, 1, 1, 1, 1.0, 2.5),      # the largest plane they take, stride 2
    (2, 10, 45, 50, 3, (3, 3), 1, 1, 1, 2, 0.6, 3.0),     # 5 tiles of 512, the last one ragged; two groups, scope 3; one sample on a grid line in fp32
    (1, 5, 112, 112, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),    # 112 x 112: wider than 64 columns, row-window staging, one 64-bit plane per workgroup in grad input
    (1, 4, 40, 130, 3, (3, 3), 1, 1, 1, 2, 0.6, 3.0),     # 130 columns: 256 lanes per staged row, two groups
    (2, 6, 112, 112, 3, (4, 4), 2, 1, 1, 1, 0.5, 8.0),    # 112 x 112 stride 2 with offsets that spread a tile's samples over most of the plane
    (1, 3, 100, 30, 3, (5, 5), 1, 1, 1, 1, 1.0, 2.5),     # narrow but taller than the 256-thread staging covers; scope 5
    (1, 20, 60, 40, 3, (4, 4), 1, 1, 1, 2, 0.7, 10.0),    # row-window grad filter: offsets of ten rows spread a tile's samples over three windows of 24 rows; two channel blocks, the second partial
    (2, 33, 56, 56, 3, (5, 5), 1, 1, 1, 1, 1.0, 2.0),     # row-window grad filter, scope 5 (two launches of 16 cells), three channel blocks
    (1, 6, 120, 100, 3, (4, 4), 1, 1, 1, 1, 0.7, 15.0),   # row-window channel-interleaved kernels (100 columns): offsets of fifteen rows, four windows of 32 rows per tile; two channel tuples
    (2, 9, 70, 96, 3, (3, 3), 1, 1, 1, 3, 0.6, 2.0),      # the same kernels in one pass: three groups of three channels, scope 3
    (1, 10, 224, 224, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),   # 224 x 224: no padded plane fits LDS; grad input in bands of 20 rows (a chunk of 8 channels and one of 2), row windows with the smaller margin
    (1, 6, 150, 200, 3, (4, 4), 2, 1, 1, 2, 0.6, 12.0),   # the band form at stride 2 with offsets of twelve rows (every band walks many tiles), two groups of three channels
    (4, 40, 56, 56, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),     # row-window grad filter with more (tile, channel block) units than persistent workgroups: 300 units on 256, runs that start and end inside a tile
    (1, 40, 112, 112, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),   # the same for the rows-and-columns-window grad filter: 98 tiles x 3 channel blocks
]
NAMES = ("forward", "grad input", "grad offset", "grad rotation", "grad filter")


def _run(case, dtype, seed=0):
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=seed, dtype=dtype)
    dev = torch.device("cuda:0")
    xg, og, rg, wg = [t.to(dev).requires_grad_() for t in (x, off, rot, wt)]
    out = deform_sample_depthwise(xg, og, rg, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"],
                                  cfg["dilation"], cfg["groups"])
    out.backward(gout.to(dev))
    torch.cuda.synchronize()
    return (x, wt, rot, off, gout, cfg), [t.detach().cpu() for t in (out, xg.grad, og.grad, rg.grad, wg.grad)]


def _oracle(inputs, np_dtype):
    x, wt, rot, off, gout, cfg = inputs
    a = [t.to(torch.float64).numpy().astype(np_dtype) for t in (x, off, rot, wt, gout)]
    out = orc.deform_sample_depthwise_forward(a[0], a[1], a[2], a[3], **cfg)
    return (out,) + tuple(orc.deform_sample_depthwise_backward(a[4], a[0], a[1], a[2], a[3], **cfg))


def assert_fp32_parity(got, o32, o64):
    assert rel_err(got[0], o32[0]) < 1e-5, NAMES[0]
    # grad input: fixed-point sums, exact on a grid of 2^-24 of the largest term or finer
    assert mixed_err(got[1], o64[1]) < 1e-5, NAMES[1]
    for i in (3, 4):
        assert rel_err(got[i], o64[i]) < 1e-4, NAMES[i]
    # The offset gradient is the slope of the bilinear patch a sample falls in, so it jumps where a
    # sampling position crosses a grid line; a position that fp32 rounds onto the line (36 + 0.9999987
    # = 37.0f) lies in the next patch than in fp64.  Each element must match one of the two oracles,
    # and all but a few the fp64 one (a few per million samples: the bound grows with the tensor).
    g = got[2].double().numpy()
    err = np.minimum(np.abs(g - o64[2]), np.abs(g - o32[2].astype(np.float64)))
    assert err.max() / np.abs(o64[2]).max() < 1e-4, NAMES[2]
    assert np.count_nonzero(np.abs(g - o64[2]) > 1e-4 * np.abs(o64[2]).max()) <= 2 + g.size // 250000, NAMES[2]


@pytest.mark.parametrize("case", CASES)
def test_fp32_matches_oracle(case):
    inputs, got = _run(case, torch.float32)
    assert_fp32_parity(got, _oracle(inputs, np.float32), _oracle(inputs, np.float64))


@pytest.mark.parametrize("case", CASES[:3])
def test_fp64_matches_oracle(case):
    inputs, got = _run(case, torch.float64)
    want = _oracle(inputs, np.float64)
    for g, w, name in zip(got, want, NAMES):
        assert rel_err(g, w) < 1e-11, name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES[:3] + [CASES[10], CASES[13], CASES[14], CASES[16], CASES[17], CASES[24], CASES[26], CASES[27]])   # planes above 30 x 30; wider than 64 columns; 224 x 224; persistent grad filter
def test_half_precisions_match_fp32_oracle(case, dtype):
    inputs, got = _run(case, dtype)
    want = _oracle(inputs, np.float32)
    for g, w, name in zip(got, want, NAMES):
        assert g.dtype == dtype
        assert rel_err(g.float(), w) < 1e-2, name


@pytest.mark.parametrize("clip", [(-0.5, 0.25), 'scope'])
@pytest.mark.parametrize("case", [CASES[0], CASES[2], CASES[4], CASES[6]])
def test_rotation_clip_inside_the_operator(case, clip):
    # the operator clamping the kernel-space offsets itself == clamping the tensor first
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, 2.0 * rs, os_, seed=7)
    dev = torch.device("cuda:0")
    xg, og, rg, wg = [t.to(dev).requires_grad_() for t in (x, off, rot, wt)]
    out = deform_sample_depthwise(xg, og, rg, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"],
                                  cfg["dilation"], cfg["groups"], clip)
    out.backward(gout.to(dev))
    got = [t.detach().cpu() for t in (out, xg.grad, og.grad, rg.grad, wg.grad)]
    rot_c, open_ = clipped_rotation(rot, clip, cfg["kernel_size"], S, G)
    assert 0.02 < 1.0 - open_.float().mean().item() < 0.9
    inputs = (x, wt, rot_c, off, gout, cfg)
    o32, o64 = _oracle(inputs, np.float32), _oracle(inputs, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5, NAMES[0]
    for i in (1, 2, 4):
        assert rel_err(got[i], o64[i]) < 1e-4, NAMES[i]
    assert rel_err(got[3], torch.as_tensor(o64[3]) * open_) < 1e-4, NAMES[3]
    assert (got[3][~open_] == 0).all()


# 14 x 14: one workgroup per output plane; 40 x 36 with 11 channels: the tiled kernel (planes above 1024 pixels:
# a plane per channel and two walks over the tiles when an element collects more than 64 samples, last chunk ragged)
@pytest.mark.parametrize("case", [(2, 12, 14, 14, 3, (4, 4), 1, 1, 1, 1, 0.5, 0.0),
                                  (1, 11, 40, 36, 3, (4, 4), 1, 1, 1, 1, 0.5, 0.0)])
def test_grad_input_when_every_sample_lands_on_one_input_element(case):
    # all 9 x P samples of an image within one input cell: the grad-input kernel's fixed-point
    # scale has to leave room for that many terms in one sum
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=9)
    g = torch.Generator().manual_seed(1)
    oh, ow = torch.meshgrid(torch.arange(H), torch.arange(W), indexing="ij")
    for t in range(9):
        # tap position oh - 1 + t // 3, ow - 1 + t % 3; target (6.3, 7.6) plus a little jitter
        off[:, 2 * t] = 6.3 - (oh - 1 + t // 3) + 0.2 * torch.rand(N, H, W, generator=g)
        off[:, 2 * t + 1] = 7.6 - (ow - 1 + t % 3) + 0.2 * torch.rand(N, H, W, generator=g)
    dev = torch.device("cuda:0")
    xg, og, rg, wg = [t_.to(dev).requires_grad_() for t_ in (x, off, rot, wt)]
    out = deform_sample_depthwise(xg, og, rg, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"],
                                  cfg["dilation"], cfg["groups"])
    out.backward(gout.to(dev))
    got = [t_.detach().cpu() for t_ in (out, xg.grad, og.grad, rg.grad, wg.grad)]
    inputs = (x, wt, rot, off, gout, cfg)
    o32, o64 = _oracle(inputs, np.float32), _oracle(inputs, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5, NAMES[0]
    assert rel_err(got[1], o64[1]) < 1e-5, NAMES[1]
    for i in range(2, 5):
        assert rel_err(got[i], o64[i]) < 1e-4, NAMES[i]


def test_zero_image_offsets_equal_the_local_operator_on_gpu():
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise, sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(2, 16, 12, 12, 3, (4, 4), 1, 1, 1, 1, 1.0, 0.0, seed=3)
    dev = torch.device("cuda:0")
    args = (cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], cfg["groups"])
    a = deform_sample_depthwise(x.to(dev), off.to(dev), rot.to(dev), wt.to(dev), *args)
    b = sample_depthwise(x.to(dev), rot.to(dev), wt.to(dev), *args)
    assert rel_err(a.cpu(), b.cpu()) < 1e-6


def test_samples_outside_the_image_give_exact_zeros():
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(1, 4, 8, 8, 3, (4, 4), 1, 1, 1, 1, 0.3, 0.0, seed=4)
    dev = torch.device("cuda:0")
    for shift in (-30.0, 30.0):
        ts = [t.to(dev).requires_grad_() for t in (x, off + shift, rot, wt)]
        out = deform_sample_depthwise(*ts, (3, 3), (1, 1), (1, 1), (1, 1), 1)
        out.backward(gout.to(dev))
        for t in [out] + [t.grad for t in ts]:
            assert torch.count_nonzero(t).item() == 0


def test_config4_shape_on_a_batch_slice():
    """benchmark configuration 4 geometry at full channel count (C=512, 28x28 -> 14x14, stride 2) on 4
    images: forward and all four gradients against the oracle."""
    case = (4, 512, 28, 28, 3, (4, 4), 2, 1, 1, 1, 0.5, 2.0)
    inputs, got = _run(case, torch.float32)
    o32, o64 = _oracle(inputs, np.float32), _oracle(inputs, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5
    for i in range(1, 5):
        assert rel_err(got[i], o64[i]) < 1e-4, NAMES[i]


def test_config4_properties_at_full_size():
    """benchmark configuration 4 (N=64, C=512, 28x28 -> 14x14, stride 2, fp32) at full size: the oracle on
    two images; the whole batch through properties that need no oracle -- the operator is linear
    in the input and in the filter, so <gout, F> = <grad_input, x> = <grad_filter, Wt>, and it is
    independent per image."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    case = (64, 512, 28, 28, 3, (4, 4), 2, 1, 1, 1, 0.5, 2.0)
    (x, wt, rot, off, gout, cfg), got = _run(case, torch.float32)
    out, gin, goff, grot, gw = got
    for n in (0, 63):
        sl = slice(n, n + 1)
        a = [t[sl].double().numpy() for t in (x, off, rot)] + [wt.double().numpy(), gout[sl].double().numpy()]
        want = orc.deform_sample_depthwise_forward(a[0], a[1], a[2], a[3], **cfg)
        w_gin, w_goff, w_grot, _ = orc.deform_sample_depthwise_backward(a[4], a[0], a[1], a[2], a[3], **cfg)
        assert rel_err(out[sl], want) < 1e-5
        assert rel_err(gin[sl], w_gin) < 1e-4
        assert rel_err(goff[sl], w_goff) < 1e-4
        assert rel_err(grot[sl], w_grot) < 1e-4
    lhs = (gout.double() * out.double()).sum().item()
    via_x = (gin.double() * x.double()).sum().item()
    via_w = (gw.double() * wt.double()).sum().item()
    assert abs(lhs - via_x) < 1e-5 * max(abs(lhs), 1.0)
    assert abs(lhs - via_w) < 1e-5 * max(abs(lhs), 1.0)
    # batch independence: images 10..13 alone give the same rows
    dev = torch.device("cuda:0")
    sl = slice(10, 14)
    with torch.no_grad():
        part = deform_sample_depthwise(x[sl].to(dev), off[sl].to(dev), rot[sl].to(dev), wt.to(dev), cfg["kernel_size"],
                                       cfg["stride"], cfg["padding"], cfg["dilation"], cfg["groups"])
    assert torch.equal(part.cpu(), out[sl])


@pytest.mark.parametrize("switch,case", [("DK_NO_DEFORM_CH", CASES[0]), ("DK_NO_DEFORM_MFMA", CASES[0]),
                                         ("DK_NO_DEFORM_CH_BIG", CASES[7]), ("DK_NO_DEFORM_WINDOW", CASES[13]),
                                         ("DK_NO_DEFORM_WINDOW", CASES[20]), ("DK_NO_DEFORM_WINDOW", CASES[16]),
                                         ("DK_NO_DEFORM_WINDOW", CASES[22]), ("DK_NO_DEFORM_WINDOW", CASES[25]),
                                         ("DK_FORCE_WIN2", CASES[13]),
                                         ("DK_FORCE_WIN2", CASES[20]), ("DK_FORCE_WIN2", CASES[21]),
                                         ("DK_FORCE_WIN2", CASES[9])])
def test_one_plane_kernels_on_a_shape_the_newer_ones_cover(switch_off, switch, case):
    """Without the channel-interleaved kernels (those for small planes and those for large ones) / the
    matrix-core grad filter / the row-window forms, the one-plane kernels serve the shape; and the grad filter with
    a window in rows and columns on shapes that its row-window form takes by default."""
    switch_off(switch)
    inputs, got = _run(case, torch.float32)
    assert_fp32_parity(got, _oracle(inputs, np.float32), _oracle(inputs, np.float64))


def test_generic_kernels_on_a_shape_the_tuned_ones_cover(switch_off):
    """With the tuned deformable kernels switched off the generic ones serve the same shape."""
    switch_off("DK_NO_DEFORM_FAST")
    inputs, got = _run(CASES[0], torch.float32)
    o32, o64 = _oracle(inputs, np.float32), _oracle(inputs, np.float64)
    assert rel_err(got[0], o32[0]) < 1e-5
    for i in range(1, 5):
        assert rel_err(got[i], o64[i]) < 1e-4, NAMES[i]


@pytest.mark.parametrize("case", [CASES[0], CASES[10], CASES[24]])  # one plane per workgroup; tiled planes above 1024 pixels; bands of rows
@pytest.mark.parametrize("poison", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["out_grad", "filter"])
def test_non_finite_values_reach_the_input_gradient(case, poison, where):
    """The tuned grad-input kernels add fixed-point integers whose scale comes from max|out_grad| and
    max|filter[c]|; an infinity or a NaN there must not come back as finite numbers (the reference's
    float atomics carry it to the elements it touches; loss scaling only asks whether any gradient
    is non-finite).  out_grad: the whole input gradient is NaN; filter: at least the poisoned
    channel's planes are, and the planes of other channel chunks stay finite."""
    from deformable_kernels.ops.deform_kernel import _lib
    L, P = _lib.lib(), _lib.ptr
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=9)
    if where == "out_grad":
        gout[N - 1, C // 2, 3, 4] = poison
    else:
        wt[1, 0, 2, 1] = poison
    dev = torch.device("cuda:0")
    wg, rg, og, gg = [t.to(dev) for t in (wt, rot, off, gout)]
    xs = torch.empty(N, C, H, W, device=dev)
    desc = _lib.conv_desc(xs, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], G)
    ws, nbytes = _lib.workspace(L.dk_deformable_sample_depthwise_backward_data_workspace(desc), dev)
    gin = torch.zeros_like(xs)
    _lib.check(L.dk_deformable_sample_depthwise_backward_data(
        desc, P(gg), P(og), P(rg), P(wg), P(gin), P(ws), nbytes, torch.cuda.current_stream().cuda_stream), "data")
    torch.cuda.synchronize()
    bad = ~torch.isfinite(gin)
    if where == "out_grad":
        assert bool(bad[N - 1, C // 2].any())   # where the reference's atomics would have put it
    else:
        assert bool(bad[:, 1].any())


# ---- no rotation tensor (DeformKernelConv2d / DeformConv2d: rotation = None) ----------------------

NO_ROTATION_CASES = [
    (2, 16, 14, 14, 3, (3, 3), 2, 1, 1, 1, 0.0, 2.0),    # DeformConv2d: scope == kernel, stride 2
    (1, 9, 56, 56, 3, (3, 3), 1, 1, 1, 1, 0.0, 2.0),     # 56 x 56 planes, the 1024-thread kernels
    (2, 12, 13, 11, 3, (4, 4), 1, 1, 1, 1, 0.0, 2.0),    # DeformKernelConv2d with a scope larger than the kernel
    (2, 6, 8, 8, (2, 3), (4, 5), (1, 2), (0, 1), 1, 3, 0.0, 1.0),  # the general kernels
    (1, 3, 5, 70, 3, (3, 3), 1, 1, 1, 1, 0.0, 1.5),      # wider than the tuned kernels take
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("case", NO_ROTATION_CASES)
def test_without_a_rotation_tensor_equals_the_oracle_with_zero_rotation(case, dtype):
    """rotation = None (a NULL pointer at the C ABI) is the reference's call with a tensor of zeros
    (ops/deform_kernel/modules/filter_sample_depthwise.py:163-168), without that tensor."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, 0.0, os_, seed=7, dtype=dtype)
    assert float(rot.abs().max()) == 0.0
    dev = torch.device("cuda:0")
    xg, og, wg = [t.to(dev).requires_grad_() for t in (x, off, wt)]
    out = deform_sample_depthwise(xg, og, None, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"],
                                  cfg["dilation"], cfg["groups"])
    out.backward(gout.to(dev))
    torch.cuda.synchronize()
    got = [t.detach().cpu() for t in (out, xg.grad, og.grad, wg.grad)]
    o64 = _oracle((x, wt, rot, off, gout, cfg), np.float64)
    want = [o64[i] for i in (0, 1, 2, 4)]
    tol = {torch.float32: (1e-5, 1e-5, 1e-4, 1e-4), torch.float64: (1e-11,) * 4, torch.bfloat16: (1e-2,) * 4}[dtype]
    for name, a, b, t in zip(("forward", "grad input", "grad offset", "grad filter"), got, want, tol):
        if name == "grad offset" and dtype == torch.float32:
            o32 = _oracle((x, wt, rot, off, gout, cfg), np.float32)[2].astype(np.float64)
            err = np.minimum(np.abs(a.double().numpy() - b), np.abs(a.double().numpy() - o32))
            assert err.max() / np.abs(b).max() < t, name
        else:
            assert rel_err(a.float() if dtype == torch.bfloat16 else a, b) < t, name


def test_deform_conv_module_runs_without_a_rotation_tensor_and_is_a_depthwise_deformable_convolution():
    """DeformConv2d (scope = kernel, rotation = None, reference modules/deform_conv.py:15-42): with
    zero image-space offsets it is the plain depthwise convolution with its own weights."""
    from deformable_kernels.modules import DeformConv2d
    dev = torch.device("cuda:0")
    torch.manual_seed(11)
    m = DeformConv2d(12, 12, kernel_size=3, stride=1, padding=1, groups=12).to(dev)
    with torch.no_grad():                                # the module marks offset_conv for zero initialisation (:262)
        m.offset_conv.weight.zero_()
        m.offset_conv.bias.zero_()
    x = torch.randn(2, 12, 10, 9, device=dev, requires_grad=True)
    out = m(x)
    want = torch.nn.functional.conv2d(x.detach().double(), m.inner_conv.weight.detach().double(), padding=1, groups=12)
    assert rel_err(out.detach().cpu(), want.cpu()) < 1e-5
    out.sum().backward()
    assert x.grad is not None and m.inner_conv.weight.grad is not None and m.offset_conv.weight.grad is not None


@pytest.mark.parametrize("case", [CASES[0], CASES[8], CASES[13]])  # one kernel (small planes, several chunks); 56 x 56: the two kernels in turn
def test_both_coordinate_gradients_from_one_call_equal_the_separate_entry_points(case):
    """dk_deformable_sample_depthwise_backward_offset_rotation forms the same sums in the same order as
    the two separate entry points, whether it runs as one kernel or as the two in turn: equal bits."""
    from deformable_kernels.ops.deform_kernel import _lib
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=3, dtype=torch.float32)
    dev = torch.device("cuda:0")
    xg, wg, rg, og, gg = [t.to(dev) for t in (x, wt, rot, off, gout)]
    L, P = _lib.lib(), _lib.ptr
    desc = _lib.conv_desc(xg, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], G)
    st = _lib.stream_ptr(xg)
    goff, grot, goff2, grot2 = [torch.empty_like(t) for t in (og, rg, og, rg)]
    ws, n = _lib.workspace(L.dk_deformable_sample_depthwise_backward_offset_workspace(desc), dev)
    _lib.check(L.dk_deformable_sample_depthwise_backward_offset(desc, P(gg), P(xg), P(og), P(rg), P(wg), P(goff), P(ws), n, st), "offset")
    ws, n = _lib.workspace(L.dk_deformable_sample_depthwise_backward_rotation_workspace(desc), dev)
    _lib.check(L.dk_deformable_sample_depthwise_backward_rotation(desc, P(gg), P(xg), P(og), P(rg), P(wg), P(grot), P(ws), n, st), "rotation")
    ws, n = _lib.workspace(L.dk_deformable_sample_depthwise_backward_offset_rotation_workspace(desc), dev)
    _lib.check(L.dk_deformable_sample_depthwise_backward_offset_rotation(
        desc, P(gg), P(xg), P(og), P(rg), P(wg), P(goff2), P(grot2), P(ws), n, st), "both")
    assert L.dk_deformable_sample_depthwise_backward_offset_rotation(
        desc, P(gg), P(xg), P(og), P(rg), P(wg), P(goff2), P(grot2), P(ws), max(n - 1, 0), st) == (-5 if n else 0)  # DK_ERR_WORKSPACE
    torch.cuda.synchronize()
    assert torch.equal(goff, goff2) and torch.equal(grot, grot2)


LANES_CASES = [
    (1, 1, 2, 3, 3, (4, 4), 1, 1, 1, 1, 0.5, 1.0),       # one channel, one unit of 16 pixels that is not full
    (2, 33, 9, 11, 3, (3, 3), 1, 1, 1, 1, 0.7, 2.0),     # 99 pixels: no group of four is aligned; a second chunk of one channel
    (1, 66, 16, 12, 3, (5, 5), 1, 1, 1, 2, 1.0, 3.0),    # two groups of 33 channels, aligned groups of four
    (1, 20, 28, 28, 3, (4, 4), 2, 1, 1, 1, 0.5, 6.0),    # stride 2, many samples outside the image
    (1, 40, 30, 31, 3, (4, 4), 1, 2, 2, 1, 0.7, 2.0),    # dilation; the largest plane whose sums fit LDS
    (1, 34, 14, 14, 3, (4, 4), 1, 1, 1, 1, 0.5, None),   # every sample in one input cell: one channel per 64-bit sum
]


def _grad_input_with_the_lanes_along_the_channels(case, dtype, rotation=True, clip=None):
    from deformable_kernels.ops.deform_kernel import _lib
    pile = case[-1] is None
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case[:-1] + (0.0,) if pile else case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=4, dtype=dtype)
    if pile:
        oh, ow = torch.meshgrid(torch.arange(H), torch.arange(W), indexing="ij")
        for t in range(9):
            off[:, 2 * t], off[:, 2 * t + 1] = 6.25 - (oh - 1 + t // 3), 7.5 - (ow - 1 + t % 3)
    if not rotation:
        rot.zero_()
    dev = torch.device("cuda:0")
    wg, rg, og, gg = [t.to(dev) for t in (wt, rot, off, gout)]
    if clip is not None:
        rot = clipped_rotation(rot, clip, cfg["kernel_size"], S, G)[0]
    gin = torch.full((N, C, H, W), float("nan"), device=dev, dtype=dtype)
    L, P = _lib.lib(), _lib.ptr
    desc = _lib.conv_desc(gin, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], G,
                          clip)
    ws, nbytes = _lib.workspace(L.dk_deformable_sample_depthwise_backward_data_workspace(desc), dev)
    with _lib.test_switches("DK_FORCE_DEFORM_LANES"):
        _lib.check(L.dk_deformable_sample_depthwise_backward_data(
            desc, P(gg), P(og), P(rg if rotation else None), P(wg), P(gin), P(ws), nbytes, _lib.stream_ptr(gin)), "grad input")
    want = _oracle((x, wt, rot, off, gout, cfg), np.float64)[1]
    if dtype == torch.float32:
        # rounding of each term on a grid of 2^-24 of the largest possible one, and of the positions
        assert mixed_err(gin.cpu(), want) < 1e-5
    else:
        assert rel_err(gin.float().cpu(), want) < 1e-2


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", LANES_CASES)
def test_grad_input_with_the_lanes_along_the_channels(case, dtype):
    _grad_input_with_the_lanes_along_the_channels(case, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", LANES_CASES)
def test_grad_input_with_the_lanes_along_the_channels_without_a_rotation_tensor(case, dtype):
    _grad_input_with_the_lanes_along_the_channels(case, dtype, rotation=False)


LANES_BAND_CASES = [
    (1, 34, 56, 56, 3, (4, 4), 1, 1, 1, 1, 0.7, 2.0),    # three bands of 19, 19 and 18 rows; a second chunk of two channels
    (2, 40, 33, 33, 3, (5, 5), 1, 1, 1, 2, 1.0, 9.0),    # the first height that needs a second band; offsets of nine rows; two groups
    (1, 18, 41, 100, 3, (4, 4), 2, 1, 1, 1, 0.5, 6.0),   # bands of ten rows and fewer at stride 2
    (1, 20, 25, 115, 3, (3, 3), 1, 2, 2, 1, 0.7, 2.0),   # bands of a few rows, dilation, rows that no group of 64 pixels ends with
    (1, 34, 56, 56, 3, (4, 4), 1, 1, 1, 1, 0.5, None),   # every sample in one cell of the first band: one channel per 64-bit sum; bands without samples
]


@pytest.mark.parametrize("rotation", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", LANES_BAND_CASES)
def test_grad_input_with_the_lanes_along_the_channels_in_bands(case, dtype, rotation):
    _grad_input_with_the_lanes_along_the_channels(case, dtype, rotation)


@pytest.mark.parametrize("rotation", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N, C, H, W, bands_of", [
    (5, 288, 56, 56, 3),    # beside the form that walks tiles of 1024 pixels
    (5, 544, 128, 8, 2),    # beside the form of one workgroup per plane
    (5, 224, 64, 64, 4),
])
def test_grad_input_in_bands_leaves_wide_offsets_to_the_form_with_a_pixel_per_lane(N, C, H, W, bands_of, dtype, rotation):
    """The default dispatch on offsets of half a pixel, of most of the plane's height, of one such image among narrow ones, and beyond
    the plane (no sample inside): the gradient is one form's to the bit -- the bands' for few rows per unit and for none -- and
    that of the oracle.  The workspace starts as garbage each time."""
    from deformable_kernels.ops.deform_kernel import _lib
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, 3, (4, 4), 1, 1, 1, 1, 0.7, 0.5, seed=6, dtype=torch.float32)
    if not rotation:
        rot.zero_()
    x, wt, rot, gout = [t.to(dtype) for t in (x, wt, rot, gout)]
    dev = torch.device("cuda:0")
    wg, rg, gg = [t.to(dev) for t in (wt, rot, gout)]
    L, P = _lib.lib(), _lib.ptr
    desc = _lib.conv_desc(x, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    ws, nbytes = _lib.workspace(L.dk_deformable_sample_depthwise_backward_data_workspace(desc), dev)

    def grad_input(og, *switches):
        gin = torch.full((N, C, H, W), float("nan"), device=dev, dtype=dtype)
        ws.fill_(0xEE)
        with _lib.test_switches(*switches):
            _lib.check(L.dk_deformable_sample_depthwise_backward_data(
                desc, P(gg), P(og), P(rg if rotation else None), P(wg), P(gin), P(ws), nbytes, _lib.stream_ptr(gin)), "grad input")
        return gin.cpu()

    # rows of offsets: per image; whether the bands take them
    always = not rotation and bands_of == 2   # without a rotation tensor two bands are never the slower form
    for rows, bands in ([1.0] * N, True), ([2.0 * H] * N, always), ([2.0 * H] + [1.0] * (N - 1), True), (None, True):
        o = off.clone()
        if rows is None:
            o += 2.5 * H
        else:
            o[:, 0::2] *= torch.tensor(rows).view(N, 1, 1, 1)
        o = o.to(dtype)
        og = o.to(dev)
        got = grad_input(og)
        assert torch.equal(got, grad_input(og, "DK_FORCE_DEFORM_LANES" if bands else "DK_NO_DEFORM_LANES"))
        want = _oracle((x, wt, rot, o, gout, cfg), np.float64)[1]
        if dtype == torch.float32:
            assert mixed_err(got, want) < 1e-5
        else:
            assert rel_err(got.float(), want) < 1e-2


@pytest.mark.parametrize("clip", [(0.25, 0.75), (-1.5, -0.75)])
def test_grad_input_with_the_lanes_along_the_channels_at_a_clipped_zero_rotation(clip):
    _grad_input_with_the_lanes_along_the_channels(LANES_CASES[2], torch.float32, rotation=False, clip=clip)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [
    (1, 1, 3, 4, 3, (4, 4), 1, 1, 1, 1, 0.0, 1.0),       # one channel, one wave that is not full
    (3, 9, 7, 7, 3, (3, 3), 1, 1, 1, 1, 0.0, 2.0),       # one channel past a step of eight; whole scope coordinates
    (2, 35, 21, 24, 3, (5, 5), 1, 1, 1, 1, 0.0, 2.0),    # 504 pixels: eight waves, the last 56 lanes; several chunks
    (1, 34, 23, 23, 3, (4, 4), 1, 2, 2, 2, 0.0, 3.0),    # 529 pixels: two tiles; two groups of 17 channels, dilation
    (1, 20, 31, 40, 3, (4, 4), 2, 1, 1, 1, 0.0, 9.0),    # stride 2, most samples outside the image
    (1, 6, 8, 120, 3, (4, 4), 4, 1, 1, 1, 0.0, 2.0),     # sixteen inputs per output: threads that only stage
    (1, 10, 57, 60, 3, (4, 4), 1, 1, 1, 1, 0.0, 2.0),    # one workgroup of 14 waves per CU, four staging passes
])
def test_without_a_rotation_tensor_on_the_kernels_of_nine_weights(case, dtype):
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, rs, os_, seed=8, dtype=dtype)
    rot.zero_()
    dev = torch.device("cuda:0")
    xg, og, wg = [t.to(dev).requires_grad_() for t in (x, off, wt)]
    out = deform_sample_depthwise(xg, og, None, wg, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], G)
    got = [out.detach()] + list(torch.autograd.grad(out, [xg, og, wg], gout.to(dev)))
    inputs = (x, wt, rot, off, gout, cfg)
    o32, o64 = _oracle(inputs, np.float32), _oracle(inputs, np.float64)
    if dtype == torch.float32:
        got.insert(3, torch.from_numpy(o64[3]))  # no rotation gradient here
        assert_fp32_parity([t.cpu() for t in got], o32, o64)
    else:
        for g, want in zip(got, (o32[0], o32[1], o32[2], o32[4])):
            assert rel_err(g.float().cpu(), want) < 1e-2


@pytest.mark.parametrize("poison", [float("inf"), float("nan")])
def test_without_a_rotation_tensor_a_tap_outside_the_image_meets_no_weight(poison):
    """A channel's weights that are not finite reach the pixels whose taps sample the image, and no others."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    g = torch.Generator().manual_seed(3)
    x, wt, off = torch.randn(1, 12, 9, 9, generator=g), torch.randn(12, 1, 4, 4, generator=g), torch.zeros(1, 18, 9, 9)
    wt[5] = poison
    off[..., :4, :] = 100.0  # the pixels of the first rows sample nothing
    xg, og, wg = [t.cuda().requires_grad_() for t in (x, off, wt)]
    out = deform_sample_depthwise(xg, og, None, wg, (3, 3), (1, 1), (1, 1), (1, 1), 1)
    goff, = torch.autograd.grad(out, og, torch.ones_like(out))
    assert (out[:, :, :4] == 0).all() and (goff[:, :, :4] == 0).all()
    assert not torch.isfinite(out[:, 5, 4:]).any() and torch.isfinite(out[:, 6:, 4:]).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rotation", [True, False])
@pytest.mark.parametrize("shape,stride,off_std", [
    ((2, 10, 9, 11), 1, 4.0),    # whole planes, interleaved
    ((1, 6, 30, 33), 2, 12.0),   # most samples outside the image
    ((1, 5, 70, 66), 1, 4.0),    # wider than 64 columns: windows of rows
])
@pytest.mark.parametrize("poison", [float("inf"), float("nan")])
def test_a_tap_outside_the_image_does_not_read_the_first_pixel(shape, stride, off_std, rotation, dtype, poison):
    """Taps that sample nothing are skipped (K.cu:500): a non-finite first pixel of a plane reaches the outputs whose
    samples touch it, and no others."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W = shape
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, 3, (4, 4), stride, 1, 1, 1, 0.5, off_std, seed=9, dtype=dtype)
    rot = rot.clamp(-1, 1) if rotation else torch.zeros_like(rot)  # (inside the scope band)
    x[:, 1::2, 0, 0] = poison
    want = orc.deform_sample_depthwise_forward(*[t.float().numpy() for t in (x, off, rot, wt)], **cfg)
    got = deform_sample_depthwise(*[t.cuda() if t is not None else None for t in (x, off, rot if rotation else None, wt)],
                                  cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    touched = ~np.isfinite(want)
    assert touched.any() and not touched.all()
    assert np.array_equal(~torch.isfinite(got).cpu().numpy(), touched)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rotation", [True, False])
@pytest.mark.parametrize("shape,stride,off_std", [
    ((2, 10, 9, 11), 1, 4.0),
    ((1, 6, 30, 33), 2, 12.0),
    ((1, 16, 20, 130), 1, 5.0),  # wider than 128 columns
])
def test_a_tap_outside_the_image_takes_no_coordinate_gradient_from_the_first_pixel(shape, stride, off_std, rotation, dtype):
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W = shape
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, 3, (4, 4), stride, 1, 1, 1, 0.5, off_std, seed=9, dtype=dtype)
    rot = rot.clamp(-1, 1) if rotation else torch.zeros_like(rot)  # (inside the scope band)
    x[:, 1::2, 0, 0] = float("nan")
    want = orc.deform_sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, off, rot, wt)], **cfg)[1:3]
    coords = [off.cuda().requires_grad_()] + ([rot.cuda().requires_grad_()] if rotation else [])
    out = deform_sample_depthwise(x.cuda(), coords[0], coords[1] if rotation else None, wt.cuda(),
                                  cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    for got, w in zip(torch.autograd.grad(out, coords, gout.cuda()), want):
        touched = ~np.isfinite(w)
        assert touched.any() and not touched.all()
        assert np.array_equal(~torch.isfinite(got).cpu().numpy(), touched)


# ---- no rotation tensor: filter gradient from the taps' sums, alone and with the offsets' gradient ----

PLAIN_FILTER_CASES = [
    (2, 1, 7, 7, 3, (3, 3), 1, 1, 1, 1, 0.0, 2.0),       # one wave, one channel
    (1, 19, 8, 8, 3, (4, 4), 1, 1, 1, 1, 0.0, 2.0),      # a full wave; channels past the last group of eight
    (2, 18, 9, 23, 3, (5, 5), 1, 1, 1, 2, 0.0, 3.0),     # two offset groups' channels interleaved, a ragged last wave
    (1, 24, 33, 31, 3, (4, 4), 2, 1, 1, 1, 0.0, 2.0),    # stride 2: the input plane in four passes of the workgroup
    (3, 12, 40, 44, 3, (3, 3), 1, 1, 1, 1, 0.0, 2.0),    # several pixel tiles
    (2, 8, 16, 12, 3, (4, 4), 1, 2, 2, 1, 0.0, 2.0),     # dilation
    (1, 48, 5, 5, 3, (3, 3), 1, 1, 1, 1, 0.0, 30.0),     # most taps outside the image
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", PLAIN_FILTER_CASES)
def test_filter_gradient_without_a_rotation_tensor(case, dtype):
    """The two ways to the filter's gradient (with the offsets' gradient in one pass, and alone) against the float64 oracle;
    the offsets' gradient against the one formed alone.  float32: a sum of P products of rounding error 2^-24 each, relative
    to a result of about the square root of P of them; 16 bit: the rounding of the result, 2^-11 and 2^-8."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, k, S, s, p, d, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, k, S, s, p, d, G, 0.0, os_, seed=9, dtype=dtype)
    args = (cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], cfg["groups"])
    og, wg = off.cuda().requires_grad_(), wt.cuda().requires_grad_()
    out = deform_sample_depthwise(x.cuda(), og, None, wg, *args)
    both = torch.autograd.grad(out, [og, wg], gout.cuda(), retain_graph=True)
    alone = [torch.autograd.grad(out, [t], gout.cuda(), retain_graph=True)[0] for t in (og, wg)]
    want = _oracle((x, wt, rot, off, gout, cfg), np.float64)[4]
    tol = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]
    assert rel_err(both[1].float().cpu(), want) < tol and rel_err(alone[1].float().cpu(), want) < tol
    assert rel_err(both[0].float().cpu(), alone[0].double().cpu().numpy()) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_an_infinite_output_gradient_of_taps_outside_the_image_reaches_no_filter(dtype):
    """The reference skips a tap outside the image (K.cu:978-984), so the output gradient of a pixel whose taps all are
    outside is multiplied with nothing."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(2, 11, 12, 10, 3, (4, 4), 1, 1, 1, 1, 0.0, 2.0, seed=3, dtype=dtype)
    args = (cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], cfg["groups"])
    off[1, :, 5, 7] = 1000.0

    def grads(value, wanted):
        gout[1, :, 5, 7] = value
        og, wg = off.cuda().requires_grad_(), wt.cuda().requires_grad_()
        out = deform_sample_depthwise(x.cuda(), og, None, wg, *args)
        return torch.autograd.grad(out, [t for t, on in zip((og, wg), wanted) if on], gout.cuda())

    for wanted in ((True, True), (False, True)):
        for a, b in zip(grads(float("inf"), wanted), grads(0.0, wanted)):
            assert torch.equal(a, b)
    gout[1, 4, 5, 7] = 0.0
    gout[0, 4, 3, 3] = float("nan")  # ... and one that is used reaches its channel's filter only
    og, wg = off.cuda().requires_grad_(), wt.cuda().requires_grad_()
    got = torch.autograd.grad(deform_sample_depthwise(x.cuda(), og, None, wg, *args), [wg], gout.cuda())[0]
    assert bool(got[4].isnan().any()) and bool(got[:4].isfinite().all()) and bool(got[5:].isfinite().all())


# one pass for the coordinates' and the filter's gradient: N, C, H, W, scope, groups, rotation std, offset std
ONE_PASS = [
    (2, 16, 7, 7, 4, 1, 0.7, 2.0),      # one tile, one block; the plane fits the window
    (5, 35, 25, 25, 4, 1, 0.7, 9.0),    # the largest such plane, ragged tiles, a block of three channels; offsets beyond it
    (3, 40, 26, 31, 3, 1, 0.7, 2.0),    # windows from the offsets; scope 3
    (2, 24, 9, 70, 4, 2, 0.7, 2.0),     # two groups of twelve channels: the offsets' gradient adds up over them
    (1, 200, 40, 36, 4, 1, 0.7, 1.0),   # thirteen blocks in shares of one: partial sums of both coordinate gradients
    (6, 176, 56, 56, 4, 1, 0.7, 2.0),   # more tiles than workgroups, eleven blocks: two shares
    (2, 20, 60, 66, 4, 1, 0.7, 6.0),    # samples spread over several windows: the separate kernels take the call
    (1, 9, 33, 35, 3, 1, 0.7, 14.0),
]


@pytest.mark.parametrize("wide_too", [False, True])
@pytest.mark.parametrize("clip", [None, (-0.5, 0.75)])
@pytest.mark.parametrize("case", ONE_PASS)
def test_coordinate_and_filter_gradients_from_one_pass(case, clip, wide_too, switch_off):
    """wide_too: without the separate kernels' channel-interleaved forms there is no choice, and calls with wide offsets walk
    their tiles in several windows."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    N, C, H, W, S, G, rs, os_ = case
    x, wt, rot, off, gout, cfg = make_deform(N, C, H, W, 3, (S, S), 1, 1, 1, G, rs, os_, seed=21)
    if wide_too:
        switch_off("DK_NO_DEFORM_CH")
    dev = torch.device("cuda:0")
    leaves = [t.to(dev).requires_grad_() for t in (x, off, rot, wt)]
    args = (cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], G)
    out = deform_sample_depthwise(*leaves, *args, clip)
    got = torch.autograd.grad(out, leaves, gout.to(dev))
    used, open_ = (rot, torch.ones_like(rot)) if clip is None else clipped_rotation(rot, clip, cfg["kernel_size"], (S, S), G)
    want = orc.deform_sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, off, used, wt)], **cfg)
    # sums of at most 9 * N * H * W products of three factors in float32, in blocks
    assert rel_err(got[1].cpu(), want[1]) < 2e-5
    assert rel_err(got[2].cpu(), torch.as_tensor(want[2]) * open_) < 2e-5
    assert rel_err(got[3].cpu(), want[3]) < 2e-5


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plain", [False, True])
def test_one_pass_in_16_bits_and_without_a_rotation_tensor(dtype, plain):
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(2, 36, 70, 90, 3, (4, 4), 1, 1, 1, 1, 0.0 if plain else 0.7, 2.0, seed=22, dtype=dtype)
    dev = torch.device("cuda:0")
    leaves = [t.to(dev).requires_grad_() for t in ((x, off, wt) if plain else (x, off, rot, wt))]
    xs, offs, rots, wts = (leaves[0], leaves[1], None, leaves[2]) if plain else leaves
    out = deform_sample_depthwise(xs, offs, rots, wts, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    got = torch.autograd.grad(out, leaves, gout.to(dev))
    want = orc.deform_sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, off, rot, wt)], **cfg)
    want = (want[0], want[1], want[3]) if plain else want
    for g, w in list(zip(got, want))[1:]:
        assert g.dtype == dtype and rel_err(g.float().cpu(), w) < (2e-3 if dtype == torch.float16 else 1e-2)  # the result's rounding


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("channels, scope", [(63, 4), (64, 4), (63, 3), (64, 3)])
def test_one_pass_on_either_side_of_64_channels(channels, scope, plain, dtype):
    """From 64 channels on one change across the cell serves both slopes."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(1, channels, 70, 90, 3, (scope, scope), 1, 1, 1, 1, 0.0 if plain else 0.7, 1.0, seed=26, dtype=dtype)
    leaves = [t.to("cuda:0").requires_grad_() for t in ((off, wt) if plain else (off, rot, wt))]
    offs, rots, wts = (leaves[0], None, leaves[1]) if plain else leaves
    out = deform_sample_depthwise(x.to("cuda:0"), offs, rots, wts, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    got = torch.autograd.grad(out, leaves, gout.to("cuda:0"))
    want = orc.deform_sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, off, rot, wt)], **cfg)
    tol = {torch.float32: 2e-5, torch.float16: 2e-3, torch.bfloat16: 1e-2}[dtype]  # sums in float32; the result's rounding
    for g, w in zip(got, (want[1], want[3]) if plain else want[1:]):
        assert g.dtype == dtype and rel_err(g.float().cpu(), w) < tol


def test_one_pass_non_finite_output_gradient_reaches_its_pixel_and_channel_only():
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(2, 24, 40, 40, 3, (4, 4), 1, 1, 1, 1, 0.5, 1.0, seed=23)
    gout[1, 17, 20, 21] = float("nan")
    leaves = [t.to("cuda:0").requires_grad_() for t in (x, off, rot, wt)]
    out = deform_sample_depthwise(*leaves, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    _, goff, grot, gw = torch.autograd.grad(out, leaves, gout.to("cuda:0"))
    for g in (goff, grot):
        bad = ~torch.isfinite(g)
        assert bad[1, :, 20, 21].all() and int(bad.sum()) == 18
    bad = ~torch.isfinite(gw)
    assert bad[17].any() and int(bad.sum()) == int(bad[17].sum())


@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("plane", [(3, 65534), (3, 65535), (3, 65536), (3, 66000), (32766, 3), (32767, 3), (32768, 3), (33100, 3)])
def test_coordinate_and_filter_gradients_of_planes_with_a_long_side(plane, plain):
    """Around the sides up to which the one-pass form holds a corner's row and column in one word."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(1, 9, *plane, 3, (4, 4), 1, 1, 1, 1, 0.0 if plain else 0.5, 1.0, seed=24)
    # coordinates that float32 holds to the last bit, 2^-7 above 2^16: none of the 10^6 samples rounds over a cell's border
    off, rot = (off * 64).round() / 64, (rot * 64).round() / 64
    leaves = [t.to("cuda:0").requires_grad_() for t in ((off, wt) if plain else (off, rot, wt))]
    offs, rots, wts = (leaves[0], None, leaves[1]) if plain else leaves
    out = deform_sample_depthwise(x.to("cuda:0"), offs, rots, wts, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
    got = torch.autograd.grad(out, leaves, gout.to("cuda:0"))
    want = orc.deform_sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, off, rot, wt)], **cfg)
    # sums of at most 2 * 10^6 products of three factors in float32, in blocks
    for g, w in zip(got, (want[1], want[3]) if plain else want[1:]):
        assert rel_err(g.cpu(), w) < 2e-5


@pytest.mark.parametrize("shape, gradient, bound", [
    # the filter's sums in pairs: 1.2 and 1.3 * 10^-7 measured, 1.9 and 2.0 with 64 partial sums in a chain
    ((16, 192, 14, 14), 2, 1.6e-7), ((8, 144, 56, 56), 2, 1.6e-7),
    # the slopes' changes across a cell from the differences on either side: 1.311 and 1.086 measured, 1.330 and 1.109 with one change for both
    ((16, 192, 28, 28), 0, 1.32e-7), ((64, 16, 20, 20), 0, 1.097e-7),
])
def test_rounding_error_of_the_gradients(shape, gradient, bound):
    """Against the operator in float64, on coordinates that float32 holds to the last bit: what the kernels' own arithmetic rounds."""
    from deformable_kernels.ops.deform_kernel.functions import deform_sample_depthwise
    x, wt, rot, off, gout, cfg = make_deform(*shape, 3, (4, 4), 1, 1, 1, 1, 0.5, 1.0, seed=25)
    off, rot = (off * 4096).round() / 4096, (rot * 4096).round() / 4096

    def grads(dtype):
        leaves = [t.to("cuda:0", dtype).requires_grad_() for t in (off, rot, wt)]
        out = deform_sample_depthwise(x.to("cuda:0", dtype), *leaves, cfg["kernel_size"], cfg["stride"], cfg["padding"], cfg["dilation"], 1)
        return torch.autograd.grad(out, leaves, gout.to("cuda:0", dtype))[gradient].double()
    got, want = grads(torch.float32), grads(torch.float64)
    assert float((got - want).norm() / want.norm()) < bound
