"""ReduceScatter layer (reference: nn/reduce_scatter.py): sums the tensors of
the workers that differ along ``axes_reduce_scatter`` and leaves every worker
its balanced slab of the sum.  Under the solo transport the absent workers
hold what the live one holds unless a gather provider supplies their tensors, so
without one the result is the live worker's slab of its own tensor times the
number of workers."""

import functools

import numpy as np
import torch

from .. import _lib
from ..utilities.torch import TensorStructure
from .module import Module


class ReduceScatter(Module):

    def __init__(self, P_x, axes_reduce_scatter=None, axes_keep=None):
        super().__init__()
        self.P_x = P_x
        if not P_x.active:
            return
        if axes_reduce_scatter is None:
            axes_reduce_scatter = [d for d in range(P_x.dim) if d not in [int(a) for a in axes_keep]]
        self.axes = tuple(int(a) for a in axes_reduce_scatter)
        self.axes_reduce_scatter = self.axes
        self.P_reducescatter = P_x.create_allreduction_partition(self.axes)
        self.identity = int(np.prod(self.P_reducescatter.shape)) == 1
        self._adjoint = _lib.Own()       # the adjoint as native nodes call it

    def forward(self, input):
        if not self.P_x.active or self.identity:
            return input
        functional = self._distdl_backend.functional.reduce_scatter
        Function = functional.ReduceScatterFunction
        if self.P_reducescatter.active and _lib.front().attachable(input):
            # The same two moves, the adjoint under a native node.
            if self._adjoint.value is None:
                self._adjoint.value = _lib.extension().Callback(functools.partial(functional.adjoint, self.P_reducescatter, self.axes))
            with torch.no_grad():
                y = functional.forward(self.P_reducescatter, self.axes, input.detach())
            return _lib.front().attach(y, input, self._adjoint.value)
        # Positional arguments as in the reference (nn/reduce_scatter.py:177-182).
        return Function.apply(input, self.P_reducescatter, TensorStructure(input), None, self.axes)
