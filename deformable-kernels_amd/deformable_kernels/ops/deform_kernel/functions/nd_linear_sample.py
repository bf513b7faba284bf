"""The N-d linear sampler with its gradients.

Same signature and layouts as the reference's ``NdLinearSampleFunction``
(``functions/nd_linear_sample.py:18-62``): ``input`` is ``[C, s_1..s_n]``,
``coord`` is ``[B, n]`` in absolute index units, the result is ``[B, C]``.
The sizes travel to the kernel as host integers (the reference builds a
device tensor per call, ``:22``) and the coordinate gradient comes back already
summed over channels (the reference sums a ``[B, n, C]`` buffer in Python,
``:48-55``).  The autograd node is native code (``csrc/dk_torch.cpp``).
"""
from .. import _lib

__all__ = ['nd_linear_sample']


class NdLinearSampleFunction:
    @staticmethod
    def apply(input, coord):
        return _lib.native().nd_linear_sample(input, coord)

    @staticmethod
    def _output_size(input, coord):
        output_size = (coord.size(0), input.size(0))
        return output_size


nd_linear_sample = NdLinearSampleFunction.apply
