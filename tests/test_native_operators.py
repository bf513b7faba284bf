"""The native operators' host path (csrc/dk_torch.cpp) where it meets the framework: transforms, threads, errors, saved
tensors.  What can be shown without a GPU runs on fake tensors or CPU tensors."""
import pytest
import torch

from deformable_kernels.ops.deform_kernel.functions import offset_conv


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
