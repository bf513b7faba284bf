"""The native operators' host path (csrc/dk_torch.cpp) where it meets the framework: transforms, threads, errors, saved
tensors.  What can be shown without a GPU runs on fake tensors or CPU tensors."""
import threading
import time

import pytest
import torch

from deformable_kernels.modules import GlobalDeformKernel2d
from deformable_kernels.ops.deform_kernel import _lib
from deformable_kernels.ops.deform_kernel.functions import image_depthwise_conv, nd_linear_sample, offset_conv


@pytest.mark.parametrize("wrapped", ["input", "weight", "neither"])
def test_offset_conv_inside_vmap_is_refused_not_returned_without_its_graph(wrapped):
    # a 29 x 29 plane: the framework's convolution serves the call, so no kernel's data pointer stops it
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x = torch.empty(3, 2, 8, 29, 29, device="cuda")
        w = torch.empty(18, 8, 3, 3, device="cuda", requires_grad=True)
        batched = torch.empty(3, 18, 8, 3, 3, device="cuda", requires_grad=True)
        calls = {"input": lambda: torch.func.vmap(lambda a: offset_conv(a, w))(x),
                 "weight": lambda: torch.func.vmap(lambda b: offset_conv(x[0], b))(batched),
                 "neither": lambda: torch.func.vmap(lambda a: a.sum() + offset_conv(x[0], w).sum())(x)}
        with pytest.raises(NotImplementedError, match="functorch"):
            calls[wrapped]()
        assert offset_conv(x[0], w).requires_grad


def test_offset_conv_takes_the_argument_forms_of_the_frameworks_convolution():
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x, w = torch.empty(2, 8, 29, 29, device="cuda"), torch.empty(18, 8, 3, 3, device="cuda")
        assert offset_conv(x, w, None, (1,), [1], (1,)).shape == (2, 18, 29, 29)  # one number in a list
        assert offset_conv(x.double(), w.double(), None, (2,), (1,), 1).shape == (2, 18, 15, 15)
        assert offset_conv(x.double(), w.double(), None, 1, "same", 1).shape == (2, 18, 29, 29)  # a named padding: float64


def test_other_python_threads_run_during_an_operator_call():
    # CPU tensors: the native entry hands them to the framework's convolution, here some 100 ms of it and more
    x, w = torch.randn(1, 64, 64, 64), torch.randn(18, 64, 3, 3)
    call = lambda: _lib.native().offset_conv(x, w, None, (1, 1), (1, 1), (1, 1), False)
    call()
    t0 = time.perf_counter()
    call()
    copies = max(1, int(0.3 / (time.perf_counter() - t0)))
    x = x.expand(copies, -1, -1, -1)
    ticks, stop = [0], threading.Event()

    def tick():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(0.001)

    thread = threading.Thread(target=tick)
    thread.start()
    try:
        before = ticks[0]
        call()
        during = ticks[0] - before
    finally:
        stop.set()
        thread.join()
    # a call that held the interpreter lock would let through a tick or two around its edges
    assert during >= 10, during


@pytest.mark.gpu
def test_failing_native_calls_raise_the_packages_error_forward_and_backward():
    # a kernel tensor whose (unused) batch stride is past what the library's 32-bit offsets take: refused on the host
    bad = torch.empty_strided((1, 8, 3, 3), (1 << 31, 1, 24, 8), device="cuda").fill_(0.5)
    x = torch.randn(1, 8, 12, 12, device="cuda", requires_grad=True)
    with pytest.raises(_lib.DkError, match="forward failed"):
        image_depthwise_conv(x, bad, 1, 1)
    good = bad.contiguous()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: bad if t.shape == bad.shape else t):
        out = image_depthwise_conv(x, good, 1, 1)
    with pytest.raises(_lib.DkError, match="grad input failed"):
        out.sum().backward()
    image_depthwise_conv(x, good, 1, 1).sum().backward()  # and the engine goes on
    assert x.grad is not None


class _Dropped(torch.autograd.Function):
    """Passes its input on, and no gradient back."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.gpu
def test_no_gradient_from_above_counts_as_zeros():
    data = torch.randn(6, 5, 5, device="cuda", requires_grad=True)
    coord = torch.rand(40, 2, device="cuda").mul_(4).requires_grad_()
    _Dropped.apply(nd_linear_sample(data, coord)).sum().backward()
    assert torch.equal(data.grad, torch.zeros_like(data)) and torch.equal(coord.grad, torch.zeros_like(coord))


@pytest.mark.gpu
def test_saved_tensor_hooks_see_everything_the_global_layer_keeps():
    torch.manual_seed(0)
    layer = GlobalDeformKernel2d((4, 4), 16, 16, 3, padding=1, groups=16).cuda()
    x = torch.randn(3, 16, 14, 14, device="cuda", requires_grad=True)
    leaves = [x] + list(layer.parameters())
    want = torch.autograd.grad(layer(x).square().sum(), leaves)
    kept = []

    def pack(t):
        kept.append(tuple(t.shape))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        out = layer(x)
    # the sampled kernels [image, tap, channel], the coordinates before and behind the clamp, the pooled input
    assert {(3, 9, 16), (2, 3, 9, 2), (3, 16), (3, 16, 14, 14)} <= set(kept), kept
    for a, b in zip(torch.autograd.grad(out.square().sum(), leaves), want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["forward replaced", "hook on every module"])
def test_the_global_layer_calls_a_linear_layer_that_is_more_than_its_parameters(how):
    torch.manual_seed(0)
    layer = GlobalDeformKernel2d((4, 4), 16, 16, 3, padding=1, groups=16).cuda()
    x, seen = torch.randn(3, 16, 14, 14, device="cuda"), []
    if how == "forward replaced":
        plain = layer.fc.forward
        layer.fc.forward = lambda v: (seen.append(layer.fc), plain(v))[1]
        layer(x)
    else:
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, args, out: seen.append(mod))
        try:
            layer(x)
        finally:
            handle.remove()
    assert any(mod is layer.fc for mod in seen)
