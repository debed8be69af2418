"""All-gather along one partitioned axis and its adjoint (reference:
backends/mpi_numpy/functional/all_gather.py:88-149, :152-230).  The collective
itself belongs to the transport; what runs here is the local re-layout the
reference does with einops (``p a b c -> a (p b) c``, zero-padding and stripping
uneven shards): the P received pieces are unpacked into their slabs of the
output by one launch of the box kernel, uneven pieces included.  The adjoint is
a reduce-scatter: every worker sums its slab of all workers' gradients in one
launch of the sum kernel (strided reads of the P slabs, one write)."""

__all__ = ["AllGatherFunction", "gather_slabs", "reduce_scatter_slabs", "single_axis"]

import functools

import numpy as np
import torch

from .... import _lib
from .... import hip_ops
from ....utilities.slicing import compute_subshape


@functools.lru_cache(maxsize=512)
def _gather_launch(local_shape, shapes, axis, elem_size):
    """(output shape, launch) that joins contiguous pieces of these shapes along
    ``axis``; the output is slot 0 of the launch, piece q slot 1 + q, and has the
    extents of ``local_shape`` off the axis, as every piece must have that is not
    empty along it.  Geometry only: a function of its arguments."""
    shape = list(local_shape)
    for piece in shapes:
        if len(piece) != len(shape) or (piece[axis] and any(n != m for d, (n, m) in enumerate(zip(piece, shape)) if d != axis)):
            raise ValueError(f"gathered piece of shape {piece} does not fit {tuple(local_shape)} along axis {axis}")
    shape[axis] = sum(s[axis] for s in shapes)
    strides = hip_ops.contiguous_strides(shape)
    entries, start = [], 0
    for q, piece in enumerate(shapes):
        entries.append((1 + q, 0, 0, start * strides[axis], piece, hip_ops.contiguous_strides(piece), strides))
        start += piece[axis]
    return tuple(shape), hip_ops.BoxLaunch(entries, elem_size)


@functools.lru_cache(maxsize=512)
def _slab(size, rank, shape, axis):
    """(shape, source slices, destination slices) of the balanced slab that
    worker ``rank`` of ``size`` keeps of a tensor along ``axis``."""
    sizes = [int(np.asarray(compute_subshape(size, r, shape[axis])).reshape(-1)[0]) for r in range(size)]
    start = sum(sizes[:rank])
    out = list(shape)
    out[axis] = sizes[rank]
    src = [slice(0, n) for n in shape]
    src[axis] = slice(start, start + sizes[rank])
    return tuple(out), src, [slice(0, n) for n in out]


def gather_slabs(P, local, axis, tag):
    """``local`` of every worker of ``P``, concatenated along ``axis`` in rank order."""
    transport = P._world.transport
    x = hip_ops.contiguous(local)
    parts = transport.gather_list(P, x, tag=tag)
    axis = range(x.dim())[axis]      # an axis the tensor has not is an IndexError
    out = _lib.front().join(x, parts, axis)
    if out is not None:
        transport.release(P, tag=tag)
        return out
    hip_ops._require_gpu(x, *parts)
    for p in parts:
        if p.dtype != x.dtype or not p.is_contiguous():
            raise ValueError(f"gathered piece {tuple(p.shape)}/{p.dtype} does not match {x.dtype} or is not contiguous")
    shape, launch = _gather_launch(tuple(x.shape), tuple([tuple(p.shape) for p in parts]), axis, x.element_size())
    out = torch.empty(shape, dtype=x.dtype, device=x.device)
    launch.run([out.data_ptr()] + [p.data_ptr() for p in parts])
    transport.release(P, tag=tag)
    return out


def reduce_scatter_slabs(P, full, axis, tag, divisor=1):
    """Sum over the workers of ``P``, in rank order, of their ``full`` tensors
    (each divided by ``divisor`` first), of which this worker keeps its balanced
    slab along ``axis``: one launch that reads the P slabs where they lie and
    writes the result once."""
    transport = P._world.transport
    g = hip_ops.contiguous(full)
    grads = transport.gather_list(P, g, tag=tag)
    axis = range(g.dim())[axis]
    shape, src, dst = _slab(int(P.size), int(P.rank), tuple(g.shape), axis)
    out = _lib.front().sum_slab(grads, axis, src[axis].start, shape[axis], divisor) if len(grads) and grads[0].shape == g.shape and \
        grads[0].dtype == g.dtype else None
    if out is not None:
        transport.release(P, tag=tag)
        return out
    out = torch.empty(shape, dtype=g.dtype, device=g.device)
    if out.numel():
        hip_ops.sum_boxes(grads, src, out, dst, divisor)
    transport.release(P, tag=tag)
    return out


def single_axis(axes, who):
    """The one tensor axis a re-layout runs along (the reference's layers pass
    a tuple of axes; its einops pattern handles one, all_gather.py:126-149)."""
    axes = [int(a) for a in np.atleast_1d(np.asarray(axes))]
    if len(axes) != 1:
        raise NotImplementedError(f"{who} along several axes is not part of this build")
    return axes[0]


class AllGatherFunction(torch.autograd.Function):
    """Positional arguments as in the reference
    (backends/mpi_numpy/functional/all_gather.py:36-37).  The tensor structures
    are accepted and not needed: the output shape follows from the gathered
    pieces.  ``P_allgather`` None stands for a gather already done by the
    caller (solo transport): only the scaling of the gradient remains."""

    @staticmethod
    def forward(ctx, input, P_allgather, input_tensor_structure, output_tensor_structure, axes, scale_backward):
        ctx.scale_backward = scale_backward
        if P_allgather is None or not P_allgather.active or P_allgather.size == 1:
            ctx.identity = True
            return input
        ctx.identity = False
        ctx.P, ctx.axis = P_allgather, single_axis(axes, "AllGather")
        return gather_slabs(P_allgather, input.detach(), ctx.axis, ("all_gather", None))

    @staticmethod
    def backward(ctx, grad_output):
        grad_output = grad_output.detach()
        # Every worker's gradient is divided before the sum (reference :188-190): the sum kernel divides as it reads.
        divisor = 1 if ctx.scale_backward is None else ctx.scale_backward
        if ctx.identity:
            return (grad_output if divisor == 1 else hip_ops.scaled(grad_output, divisor)), None, None, None, None, None
        dx = reduce_scatter_slabs(ctx.P, grad_output, ctx.axis, ("all_gather_adjoint", None), divisor)
        return dx, None, None, None, None, None
