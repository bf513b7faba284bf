"""The gradients of small layers, computed in one launch (dk_local_small.hip), against the float64 oracle: every sum is
float32 over at most 256 channels or 2048 pixels x 9 taps in parts of at most 18 terms per lane, so the parity bars of the
larger kernels hold (1e-5 grad input, 1e-4 the reductions, 1e-2 for 16-bit tensors)."""
import pytest
import torch

from _cases import make_local, rel_err
from oracle import dk_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _supported(cfg, shape, scope, dtype_name, layout):
    from deformable_kernels.ops.deform_kernel import _lib
    N, C, H, W = shape
    k, s, p, d = (cfg[n] for n in ("kernel_size", "stride", "padding", "dilation"))
    desc = _lib.ConvDesc(N, C, H, W, *k, *s, *p, *d, *scope, cfg["groups"], {"float32": 0, "float16": 1, "bfloat16": 2}[dtype_name])
    desc.layout = layout
    return _lib.lib().dk_sample_depthwise_backward_workspace(desc) == 0


# N, C, H, W, scope, stride, padding, dilation, groups
CASES = [
    (2, 32, 28, 28, 4, 1, 1, 1, 1),     # the benchmark's small layer
    (1, 1, 1, 1, 3, 1, 1, 1, 1),        # one pixel, one channel: 63 lanes and 15 waves without work
    (1, 17, 8, 8, 4, 1, 1, 1, 1),       # exactly one tile of 64 pixels; one channel more than waves
    (5, 66, 5, 13, 5, 1, 1, 1, 2),      # 325 pixels, two groups of 33 channels (two shares of the channels, one short)
    (2, 256, 32, 32, 4, 1, 1, 1, 1),    # the largest: 2048 pixels, 256 channels
    (2, 48, 48, 8, 3, 1, 1, 1, 1),
    (3, 40, 9, 11, 7, 1, 1, 1, 1),      # 64 table blocks: all lanes stage
    (1, 17, 56, 56, 5, 2, 1, 1, 1),     # stride 2, even and ...
    (2, 24, 15, 17, 4, 2, 1, 1, 3),     # ... odd planes, three groups
    (2, 16, 12, 20, 4, 1, 0, 2, 1),     # no padding, dilation 2
    (2, 16, 12, 20, 4, 3, 2, 1, 16),    # stride 3, padding 2, a group per channel
]


@pytest.mark.parametrize("layout", ["planar", "channels_last"])
@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("case", CASES)
def test_gradients_of_small_layers_in_one_launch(case, dtype_name, layout):
    from deformable_kernels.ops.deform_kernel.functions import sample_depthwise
    N, C, H, W, S, s, p, d, G = case
    dtype = getattr(torch, dtype_name)
    x, wt, rot, gout, cfg = make_local(N, C, H, W, 3, (S, S), s, p, d, G, 1.0, seed=5)
    x, wt, rot, gout = [t.to(dtype) for t in (x, wt, rot, gout)]
    if layout == "planar":
        assert _supported(cfg, (N, C, H, W), (S, S), dtype_name, 0)
    fmt = torch.contiguous_format if layout == "planar" else torch.channels_last
    xg, rg, wg = [t.to(DEV).requires_grad_() for t in (x.contiguous(memory_format=fmt), rot.contiguous(memory_format=fmt), wt)]
    out = sample_depthwise(xg, rg, wg, *(cfg[k] for k in ("kernel_size", "stride", "padding", "dilation", "groups")))
    out.backward(gout.to(DEV).contiguous(memory_format=fmt))
    want = orc.sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, rot, wt)], **cfg)
    again = torch.autograd.grad(sample_depthwise(xg, rg, wg, *(cfg[k] for k in ("kernel_size", "stride", "padding", "dilation", "groups"))),
                                (xg, rg, wg), gout.to(DEV).contiguous(memory_format=fmt))
    for got, rep, ref, tol in zip((xg.grad, rg.grad, wg.grad), again, want, (1e-5, 1e-4, 1e-4)):
        assert rel_err(got.double().cpu(), ref) < (tol if dtype_name == "float32" else 1e-2)
        assert torch.equal(got, rep)   # fixed order of every sum


@pytest.mark.parametrize("clip", ["scope", (-0.4, 0.3)])
def test_clipped_offsets_and_single_gradients(clip):
    """The operator's own clamp, and each gradient asked for by itself: the same numbers as the larger kernels' (a test
    switch takes the one-launch form away) within 1e-5."""
    from deformable_kernels.ops.deform_kernel import _lib
    from deformable_kernels.ops.deform_kernel.modules import SampleDepthwise
    torch.manual_seed(3)
    m = SampleDepthwise((4, 4), 24, 24, kernel_size=3, stride=1, padding=1, groups=24).to(DEV)
    x = torch.randn(2, 24, 13, 9, device=DEV, requires_grad=True)
    r = torch.randn(2, 18, 13, 9, device=DEV, requires_grad=True)
    g = torch.randn(2, 24, 13, 9, device=DEV)
    leaves = (x, r, m.weight)
    res = torch.autograd.grad(m(x, r, clip), leaves, g)
    for k, leaf in enumerate(leaves):
        assert torch.equal(torch.autograd.grad(m(x, r, clip), (leaf,), g)[0], res[k])
    with _lib.test_switches("DK_NO_IMAGE_FLAT"):
        ref = torch.autograd.grad(m(x, r, clip), leaves, g)
    for a, b in zip(res, ref):
        assert rel_err(a.cpu(), b.cpu()) < 1e-5
    assert torch.equal(res[1] == 0, ref[1] == 0)   # where the clamp is active


# ---- values that are not finite: the default dispatch against the oracle's own NaN and Inf ----

NON_FINITE = {
    "weight, first cell": lambda x, wt, rot, gout: wt[5, 0].__setitem__((0, 0), float("inf")),
    "weight, inner cell": lambda x, wt, rot, gout: wt[5, 0].__setitem__((1, 2), float("nan")),
    "output gradient": lambda x, wt, rot, gout: gout[1, 4].__setitem__((2, 3), float("inf")),
    "input": lambda x, wt, rot, gout: x[1, 4].__setitem__((4, 5), float("inf")),
    "output gradient of a corner pixel": lambda x, wt, rot, gout: gout[0, 4].__setitem__((0, 0), float("nan")),
}


@pytest.mark.parametrize("layout", ["planar", "channels_last"])
@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("S, stride, G", [(3, 1, 1), (4, 1, 1), (4, 2, 1), (5, 1, 2), (7, 2, 1)])
@pytest.mark.parametrize("what", NON_FINITE)
def test_a_non_finite_value_reaches_what_the_reference_lets_it_reach(what, S, stride, G, dtype_name, layout):
    """No test switch is set.  Taps outside the image or the scope and, at stride 2, off its grid read nothing of the channel
    with the poisoned value, and a product reaches the four cells of its own sample."""
    from deformable_kernels.ops.deform_kernel.functions import sample_depthwise
    x, wt, rot, gout, cfg = make_local(2, 16, 11, 13, 3, (S, S), stride, 1, 1, G, 0.7, seed=8)
    rot[0, :, 1, 1] = 50.0   # all taps of this pixel leave the scope
    x, wt, rot, gout = [t.to(getattr(torch, dtype_name)) for t in (x, wt, rot, gout)]
    NON_FINITE[what](x, wt, rot, gout)
    fmt = torch.contiguous_format if layout == "planar" else torch.channels_last
    leaves = [t.to(DEV).requires_grad_() for t in (x.contiguous(memory_format=fmt), rot.contiguous(memory_format=fmt), wt)]
    out = sample_depthwise(*leaves, *(cfg[k] for k in ("kernel_size", "stride", "padding", "dilation", "groups")))
    got = torch.autograd.grad(out, leaves, gout.to(DEV).contiguous(memory_format=fmt))
    want = orc.sample_depthwise_backward(*[t.double().numpy() for t in (gout, x, rot, wt)], **cfg)
    # (that input gradient is the table kernel's, whose dead taps meet the first cell)
    table = layout == "channels_last" and dtype_name == "float32" and stride == 2 and what == "weight, first cell"
    for name, a, b in list(zip(("input", "rotation", "filter"), got, want))[1 if table else 0:]:
        finite = torch.from_numpy(b).isfinite()
        assert torch.equal(a.cpu().isfinite(), finite), name
        assert rel_err(a.cpu().double()[finite], b[finite.numpy()]) < (1e-5 if dtype_name == "float32" else 1e-2), name


@pytest.mark.parametrize("case", [
    (2, 40, 20, 20, (4, 4), 1, 2),
    (2, 96, 15, 18, (3, 3), 1, 2),
    (1, 17, 33, 31, (5, 5), 1, 3),
    (2, 24, 16, 14, (4, 4), 3, 2),   # three groups
])
def test_float32_channels_last_grad_input_above_stride_1_is_the_table_kernels_to_the_bit(case):
    """Alone, with the other gradients in their one launch, and with the kernels of the larger layers."""
    from deformable_kernels.ops.deform_kernel import _lib
    from deformable_kernels.ops.deform_kernel.functions import sample_depthwise
    N, C, H, W, S, G, s = case
    x, wt, rot, gout, cfg = make_local(N, C, H, W, 3, S, s, 1, 1, G, 0.5, seed=4)
    cl = torch.channels_last
    leaves = [t.to(DEV).requires_grad_() for t in (x.contiguous(memory_format=cl), rot.contiguous(memory_format=cl), wt)]
    gout = gout.to(DEV).contiguous(memory_format=cl)

    def grads(wanted):
        out = sample_depthwise(*leaves, *(cfg[k] for k in ("kernel_size", "stride", "padding", "dilation", "groups")))
        return torch.autograd.grad(out, wanted, gout)

    small = grads(leaves)
    with _lib.test_switches("DK_NO_NHWC_MFMA"):
        table = grads(leaves)
    assert torch.equal(small[0], table[0]) and torch.equal(grads(leaves[:1])[0], table[0])
    for a, b in zip(small[1:], table[1:]):
        assert rel_err(a.cpu(), b.double().cpu().numpy()) < 1e-5


@pytest.mark.parametrize("one_launch, shape, scope, stride, G, dtype_name, channels_last", [
    (True, (2, 32, 28, 28), 4, 1, 1, "float32", False), (True, (2, 256, 32, 32), 7, 1, 1, "bfloat16", False),
    (True, (2, 512, 32, 32), 4, 1, 2, "float32", False), (True, (1, 512, 28, 28), 4, 1, 8, "float32", False),
    (False, (1, 512, 28, 28), 4, 1, 16, "bfloat16", False), (False, (2, 256, 32, 32), 4, 1, 16, "float32", False),
    (False, (2, 1024, 32, 32), 4, 1, 4, "float32", False), (False, (1, 4096, 7, 7), 7, 1, 16, "float32", False),
    (False, (2, 256, 32, 33), 4, 1, 1, "float32", False), (False, (1, 257, 7, 7), 4, 1, 1, "float32", False),
    (True, (2, 32, 32, 32), 4, 1, 1, "float32", True), (False, (2, 40, 32, 32), 4, 1, 1, "bfloat16", True),
    (True, (2, 16, 56, 56), 4, 2, 1, "float32", True), (False, (2, 24, 56, 56), 4, 2, 1, "float32", True),
    (True, (2, 24, 56, 56), 4, 2, 1, "float16", True), (True, (2, 128, 32, 32), 7, 1, 1, "float32", True),
    (False, (2, 136, 32, 32), 7, 1, 1, "float32", True), (True, (2, 132, 32, 32), 4, 1, 1, "float32", True),
    (True, (2, 64, 32, 32), 4, 1, 2, "bfloat16", True),
])
def test_layers_that_take_the_one_launch(one_launch, shape, scope, stride, G, dtype_name, channels_last):
    """Either side of the rule's lines (channels-last too, where the gradients' own tests cannot tell the route)."""
    cfg = {"kernel_size": (3, 3), "stride": (stride,) * 2, "padding": (1, 1), "dilation": (1, 1), "groups": G}
    assert _supported(cfg, shape, (scope, scope), dtype_name, int(channels_last)) == one_launch
