"""Repartition forward / adjoint on one GPU.

Order of operations follows the reference
(backends/mpi_numpy/functional/repartition.py:142-213 forward, :285-355
adjoint): pack every outgoing overlap into its contiguous buffer, hand the
buffers to the transport, create the output, copy the self overlap directly,
unpack every incoming buffer.  The differences are where the work runs: all
outgoing boxes are packed by ONE kernel launch, which also makes the self copy,
and all incoming boxes are unpacked by ONE launch (``ddl_copy_boxes`` on box
descriptors that are built once per input structure, where the reference
builds its overlap lists) instead of one strided copy per peer, and the output
is not zero-filled first when the incoming boxes tile it completely (they
always do for a valid pair of partitions).
"""

__all__ = ["RepartitionFunction", "native_repartition"]

import functools

import numpy as np
import torch

from .... import _lib
from .... import hip_ops
from ....utilities.torch import zero_volume_tensor
from .. import buffer as _buffer
from ..transport import SoloTransport

_FWD_TAG = 111
_ADJ_TAG = 113


class OverlapList(list):
    """List of ``(slices, shape, partner)`` that also carries the C descriptors
    derived from it, so that they are built once per input structure."""

    def __init__(self, *args):
        super().__init__(*args)
        self.plans = {}


def _plan(overlaps, tensor, which):
    """Box plan of the non-self (``which='remote'``) overlaps of ``tensor``."""
    cache = getattr(overlaps, "plans", None)
    key = (which, tuple(tensor.shape), tuple(tensor.stride()))
    if cache is not None and key in cache:
        return cache[key]
    boxes = []
    for sl, sh, partner in overlaps:
        if sl is None or partner == "self":
            boxes.append(None)
        else:
            boxes.append(sl)
    plan = hip_ops.BoxPlan.from_slices(tensor, boxes)
    if cache is not None:
        cache[key] = plan
    return plan


def _views(overlaps, buffers):
    out = []
    for (sl, sh, partner), buff in zip(overlaps, buffers):
        out.append(None if buff is None else buff.get_view(sh))
    return out


def _self_slices(overlaps):
    for sl, sh, partner in overlaps:
        if partner == "self":
            return sl
    return None


def _covered(overlaps, shape):
    """Do the (disjoint) overlaps tile a tensor of this shape completely?"""
    cache = getattr(overlaps, "plans", None)
    key = ("covered", shape)
    if cache is not None and key in cache:
        return cache[key]
    volume = 0
    for sl, sh, partner in overlaps:
        if sl is not None:
            volume += int(np.prod(sh, dtype=np.int64))
    covered = volume == int(np.prod(shape, dtype=np.int64))
    if cache is not None:
        cache[key] = covered
    return covered


_SRC, _OUT, _FIXED = 0, 1, 2     # base addresses of a launch: the source tensor, the output, 0 (buffers, by their address)


class _MovePlan:
    """One direction of a Repartition (x -> y, or dy -> dx) for one input
    structure, lowered once to the two launches it takes:

      first   every outgoing box packed into its send buffer, and the box this
              worker keeps copied straight into the output
      second  every receive buffer unpacked into the output

    The box descriptors are built here; a call only adds the addresses that
    change (the source tensor, the fresh output).  Buffer views have
    fixed addresses until some pooled buffer is reallocated, which invalidates
    the plan (``stale``).
    """

    def __init__(self, src, dtype, src_active, src_overlaps, src_buffers, dst_active, dst_overlaps, dst_buffers, dst_shape):
        self.reallocations = _buffer.reallocations()
        self.elem_size = torch.empty((), dtype=dtype).element_size()
        if src_active and src.dtype != dtype:
            raise ValueError(f"Repartition was set up for {dtype}, got a tensor of {src.dtype}")
        self.send_views = _views(src_overlaps, src_buffers) if src_active else []
        self.recv_views = _views(dst_overlaps, dst_buffers) if dst_active else []
        self.keep = (src_overlaps, src_buffers, dst_overlaps, dst_buffers)     # ids of these are part of the cache key
        self.out_shape = None if dst_shape is None else tuple(int(n) for n in dst_shape)
        self.zero_fill = dst_active and not _covered(dst_overlaps, self.out_shape)
        src_strides = [int(v) for v in src.stride()]
        out_strides = hip_ops.contiguous_strides(self.out_shape) if dst_active else None

        def offset(slices, strides):
            return sum(int(sl.start) * st for sl, st in zip(slices, strides))

        def at(view):
            return view.data_ptr() // self.elem_size      # in elements from address 0; views start at a multiple of their elements

        first, second = [], []
        if src_active:
            for (sl, sh, partner), view in zip(src_overlaps, self.send_views):
                if view is not None and view.numel() > 0:
                    shape = [int(n) for n in sh]
                    first.append((_SRC, offset(sl, src_strides), _FIXED, at(view), shape, src_strides, hip_ops.contiguous_strides(shape)))
            s_self, d_self = _self_slices(src_overlaps), (_self_slices(dst_overlaps) if dst_active else None)
            if s_self is not None and d_self is not None:
                shape = [int(sl.stop) - int(sl.start) for sl in s_self]
                if int(np.prod(shape, dtype=np.int64)) > 0:
                    first.append((_SRC, offset(s_self, src_strides), _OUT, offset(d_self, out_strides), shape, src_strides, out_strides))
        if dst_active:
            for (sl, sh, partner), view in zip(dst_overlaps, self.recv_views):
                if view is not None and view.numel() > 0:
                    shape = [int(n) for n in sh]
                    second.append((_FIXED, at(view), _OUT, offset(sl, out_strides), shape, hip_ops.contiguous_strides(shape), out_strides))
        self.first = hip_ops.BoxLaunch(first, self.elem_size)
        self.second = hip_ops.BoxLaunch(second, self.elem_size)
        self.sends = [(partner, view) for (sl, sh, partner), view in zip(src_overlaps, self.send_views) if view is not None] \
            if src_active else []
        self.recvs = [(partner, view) for (sl, sh, partner), view in zip(dst_overlaps, self.recv_views) if view is not None] \
            if dst_active else []

    def stale(self):
        return self.reallocations != _buffer.reallocations()


def _move_plan(src, dtype, P_src, src_overlaps, src_buffers, P_dst, dst_overlaps, dst_buffers, dst_shape):
    cache = getattr(src_overlaps, "plans", None)
    if cache is None:
        cache = getattr(dst_overlaps, "plans", None)
    key = ("move", src.shape, src.stride(), src.dtype, dtype, id(src_overlaps), id(src_buffers), id(dst_overlaps),
           id(dst_buffers), None if dst_shape is None else tuple(int(n) for n in dst_shape))
    plan = None if cache is None else cache.get(key)
    if plan is None or plan.stale():
        plan = _MovePlan(src, dtype, P_src.active, src_overlaps, src_buffers, P_dst.active, dst_overlaps, dst_buffers, dst_shape)
        if cache is not None:
            cache[key] = plan
    return plan


def _move(src, P_union, dtype, P_src, src_overlaps, src_buffers, P_dst, dst_overlaps, dst_buffers, dst_shape,
          preserve_batch, tag):
    """Shared body of forward (x -> y) and adjoint (dy -> dx)."""
    device = src.device
    if not (P_src.active or P_dst.active):
        if preserve_batch:
            return zero_volume_tensor(src.shape[0], dtype=dtype, device=device)
        return zero_volume_tensor(dtype=dtype, device=device)
    if P_src.active and not src.is_cuda:
        raise RuntimeError(f"distdl_amd: tensor on {src.device}; the HIP path only accepts GPU tensors and there is "
                           "no CPU fallback")

    plan = _move_plan(src, dtype, P_src, src_overlaps, src_buffers, P_dst, dst_overlaps, dst_buffers, dst_shape)
    if P_dst.active:
        alloc = torch.zeros if plan.zero_fill else torch.empty
        out = alloc(plan.out_shape, dtype=dtype, device=device)
        out_ptr = out.data_ptr()
    else:
        out = zero_volume_tensor(src.shape[0], dtype=dtype, device=device) if preserve_batch else \
            zero_volume_tensor(dtype=dtype, device=device)
        out_ptr = 0
    bases = [src.data_ptr() if P_src.active else 0, out_ptr, 0]
    plan.first.run(bases)
    if P_union.active and (plan.sends or plan.recvs):
        P_union._world.transport.exchange(P_union, [(p, v, tag) for p, v in plan.sends],
                                          [(p, v, tag) for p, v in plan.recvs])
    plan.second.run(bases)
    return out


def _adjoint(P_union, dtype, P_y, P_y_to_x_overlaps, P_y_to_x_buffers, P_x, P_x_to_y_overlaps, P_x_to_y_buffers, x_shape, preserve_batch,
             grad_output):
    """The same movement with the two overlap lists exchanged; the boxes are disjoint, so it copies and never adds
    (reference :344-346)."""
    return _move(grad_output.detach(), P_union, dtype, P_y, P_y_to_x_overlaps, P_y_to_x_buffers, P_x, P_x_to_y_overlaps, P_x_to_y_buffers,
                 x_shape, preserve_batch, _ADJ_TAG)


def native_repartition(input, P_union, x_global_structure, x_local_structure, y_local_structure, P_x, P_x_to_y_overlaps, P_x_to_y_buffers,
                       P_y, P_y_to_x_overlaps, P_y_to_x_buffers, preserve_batch):
    """Forward and, if it requires gradients, adjoint for tensors like ``input`` as native moves, where no message is sent
    between their launches: the live rank of a solo transport that is in both partitions.  None otherwise."""
    dtype = x_global_structure.dtype
    if not (P_union.active and P_x.active and P_y.active and type(P_union._world.transport) is SoloTransport and input.is_cuda) or \
       input.dtype != dtype:
        return None
    x_shape, y_shape = tuple(int(n) for n in x_local_structure.shape), tuple(int(n) for n in y_local_structure.shape)
    if tuple(input.shape) != x_shape:
        return None
    general = functools.partial(_adjoint, P_union, dtype, P_y, P_y_to_x_overlaps, P_y_to_x_buffers, P_x, P_x_to_y_overlaps, P_x_to_y_buffers,
                                x_local_structure.shape, preserve_batch)
    out, epoch = [None, None], _lib.buffers_epoch()
    directions = [(input, y_shape, None, (P_x, P_x_to_y_overlaps, P_x_to_y_buffers, P_y, P_y_to_x_overlaps, P_y_to_x_buffers))]
    if input.requires_grad:
        directions.append((torch.empty(y_shape, dtype=dtype, device="meta"), x_shape, general,
                           (P_y, P_y_to_x_overlaps, P_y_to_x_buffers, P_x, P_x_to_y_overlaps, P_x_to_y_buffers)))
    for i, (src, shape, back, args) in enumerate(directions):
        plan = _move_plan(src, dtype, *args, shape)
        views = plan.send_views + plan.recv_views
        if plan.zero_fill or any(v is not None and not v.is_cuda for v in views):
            return None
        # slot 2 is address 0: the plan's boxes name their buffers by address, and the buffers stay with the object
        out[i] = hip_ops.native_moves(epoch, src, shape, [(plan.first, _lib.DDL_OP_COPY, _lib.DDL_DT_BITS),
                                                          (plan.second, _lib.DDL_OP_COPY, _lib.DDL_DT_BITS)], [None] + views, general=back)
    return out


class RepartitionFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, input, P_union, x_global_structure,
                x_local_structure, y_local_structure,
                P_x, P_x_to_y_overlaps, P_x_to_y_buffers,
                P_y, P_y_to_x_overlaps, P_y_to_x_buffers, preserve_batch):
        ctx.P_union = P_union
        ctx.x_global_structure = x_global_structure
        ctx.x_local_structure = x_local_structure
        ctx.P_x = P_x
        ctx.P_x_to_y_overlaps = P_x_to_y_overlaps
        ctx.P_x_to_y_buffers = P_x_to_y_buffers
        ctx.P_y = P_y
        ctx.P_y_to_x_overlaps = P_y_to_x_overlaps
        ctx.P_y_to_x_buffers = P_y_to_x_buffers
        ctx.preserve_batch = preserve_batch
        ctx.device = input.device

        # The reference shares requires_grad of the first input worker with the
        # whole union on every call (repartition.py:111-127).
        rg = input.requires_grad
        if P_union.active:
            rg = bool(P_union.broadcast_data(bool(input.requires_grad) if P_x.active else None, root=0))
        ctx.input_requires_grad = rg

        return _move(input.detach(), P_union, x_global_structure.dtype,
                     P_x, P_x_to_y_overlaps, P_x_to_y_buffers,
                     P_y, P_y_to_x_overlaps, P_y_to_x_buffers,
                     y_local_structure.shape if P_y.active else None, preserve_batch, _FWD_TAG)

    @staticmethod
    def backward(ctx, grad_output):
        grad_input = _adjoint(ctx.P_union, ctx.x_global_structure.dtype,
                              ctx.P_y, ctx.P_y_to_x_overlaps, ctx.P_y_to_x_buffers,
                              ctx.P_x, ctx.P_x_to_y_overlaps, ctx.P_x_to_y_buffers,
                              ctx.x_local_structure.shape if ctx.P_x.active else None, ctx.preserve_batch, grad_output)
        return grad_input, None, None, None, None, None, None, None, None, None, None, None
