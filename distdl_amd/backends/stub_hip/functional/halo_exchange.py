"""HaloExchange forward / adjoint on one GPU.

Dimension-ordered exchange of the reference
(backends/mpi_numpy/functional/halo_exchange.py:13-78 forward, :81-144
adjoint).  Per exchange dimension the two bulk slabs are packed by one launch (the first
dimension's by the launch that copies the input, the next ones' by the launch that
unpacks), the transport swaps them with the neighbours, and the two ghost slabs are
unpacked by one launch; dimension i sees the ghosts of dimensions < i, which is what
makes the corners right: those of dimension i - 1 it takes from the buffers they are
being unpacked from.  The
adjoint walks the dimensions backwards: move the ghosts out (pack and clear, one
launch), swap, ADD what arrives into the bulk.
"""

__all__ = ["HaloExchangeFunction", "native_exchange"]

import functools
import math
import operator

import torch

from .... import _lib
from .... import hip_ops
from ....utilities.slicing import compute_nd_slice_shape
from ....utilities.torch import zero_volume_tensor
from ..partition import PROC_NULL
from ..transport import SoloTransport

_LTAG = 0
_RTAG = 1


class SliceTable(list):
    """The per-dimension ``[left bulk, left ghost, right bulk, right ghost]``
    slices plus the C descriptors derived from them."""

    def __init__(self, *args):
        super().__init__(*args)
        self.plans = {}


_INPUT, _TENSOR = 0, 1     # slots of a launch's base addresses; buffer j of dimension i has 2 + 4 i + j
_LEFT_BULK, _LEFT_GHOST, _RIGHT_BULK, _RIGHT_GHOST = range(4)


class _Plan:
    """The launches of one direction for one structure of the tensor, lowered
    once, for the first ``dims`` dimensions (those of the partition).
    ``present[i][j]`` says whether strip ``j`` of dimension ``i`` has a buffer.  What is kept is geometry only: the buffers are those of the call
    (and a pooled buffer may have been reallocated since the last one)."""

    def __init__(self, dims, slices, present, shape, strides, elem_size, forward):
        self.dims = []
        tensor_strides = hip_ops.contiguous_strides(shape)

        def boxes(i, sides, to_buffer, from_input=False):
            """Boxes between the strips ``sides`` of dimension ``i`` and their buffers."""
            out = []
            for j in sides:
                if not present[i][j]:
                    continue
                start, stop = [int(s.start) for s in slices[i][j]], [int(s.stop) for s in slices[i][j]]
                extent = list(map(operator.sub, stop, start))
                if min(start) < 0 or min(extent) < 0 or any(map(operator.gt, stop, shape)):
                    # a shard narrower than its strips; the copies know no extents
                    raise RuntimeError(f"halo strip {j} of dim {i}, {list(zip(start, stop))}, is outside extents {tuple(shape)}")
                own = strides if from_input else tensor_strides
                offset = sum(map(operator.mul, start, own))
                packed = hip_ops.contiguous_strides(extent)
                slot = 2 + 4 * i + j
                if to_buffer:
                    out.append((_INPUT if from_input else _TENSOR, offset, slot, 0, extent, own, packed))
                else:
                    out.append((slot, 0, _TENSOR, offset, extent, packed, own))
            return out

        bulk, ghost = (_LEFT_BULK, _RIGHT_BULK), (_LEFT_GHOST, _RIGHT_GHOST)
        # The copy of the input takes the strips of the first dimension that sends any along: nothing has been written over
        # them yet, and no other dimension's strips are in the buffers, which all dimensions share.
        first = [(_INPUT, 0, _TENSOR, 0, list(shape), strides, tensor_strides)]
        untouched, previous = True, []
        for i in range(dims):
            extents = [tuple(int(n) for n in compute_nd_slice_shape(s)) for s in slices[i]]
            if forward:
                pack, unpack = boxes(i, bulk, True, untouched), boxes(i, ghost, False)
                merged = untouched
                untouched = untouched and not pack and not unpack
                if merged:
                    first += pack
                    pack = []
                # The ghosts of the dimension before are unpacked by the launch that packs this one's strips.
                both = self._with_unpacking(previous, pack, i, slices, present) if previous and pack else None
                self.dims.append((extents, hip_ops.BoxLaunch(pack, elem_size), hip_ops.BoxLaunch(unpack, elem_size),
                                  hip_ops.BoxLaunch(both, elem_size) if both else None))
                previous = unpack
            else:
                add = boxes(i, bulk, False)
                if len(add) == 2 and slices[i][0][i].stop > slices[i][2][i].start:
                    # Narrow shards: the left and right bulk strips share elements, so
                    # the two accumulations must not run in one launch.
                    adds = [hip_ops.BoxLaunch(add[:1], elem_size), hip_ops.BoxLaunch(add[1:], elem_size)]
                else:
                    adds = [hip_ops.BoxLaunch(add, elem_size)]
                out = hip_ops.BoxLaunch(boxes(i, ghost, True), elem_size)
                left, right = slices[i][_LEFT_GHOST], slices[i][_RIGHT_GHOST]
                clear = None
                # A ghost leaves and is cleared in one launch.  Not where the two share elements (one box would read what
                # the other has cleared), nor where a ghost has no buffer and is cleared all the same.
                if out.n and (left[i].stop > right[i].start or any(not present[i][j] and min(extents[j]) > 0 for j in ghost)):
                    clear = hip_ops.BoxPlan(shape, strides, [([int(s.start) for s in b], [int(s.stop) - int(s.start) for s in b])
                                                             for b in (left, right)])
                self.dims.append((extents, out, clear, adds))
        self.first = hip_ops.BoxLaunch(first, elem_size) if forward else None
        self.adds = any(present[i][j] for i in range(dims) for j in bulk)

    @staticmethod
    def _with_unpacking(unpack, pack, i, slices, present):
        """The boxes ``unpack`` of dimension ``i - 1`` and ``pack`` of dimension ``i`` as those of one launch: what a strip
        has in a ghost comes from that ghost's buffer instead of from the tensor.  None where strips reach out of what the
        buffers hold, or where the ghosts share elements; nor for many rows of strips along the innermost dimension, whose
        launch of their own has the two strips of a row on one XCD (66 thousand rows of one fp32: two launches 11.9 us, one
        8.4; 606 thousand: 30, one 43.  A whole exchange around the line: 66 thousand rows 28.5 and 28.1, 102 thousand 47.3 and
        49.3 in two dimensions, 33.8 and 32.0 in three, 131 thousand 69.6 and 70.6, 262 thousand 81 and 88)."""
        p = i - 1
        left, right = slices[p][_LEFT_GHOST], slices[p][_RIGHT_GHOST]
        if left[p].stop > right[p].start:
            return None
        if i == len(left) - 1 and math.prod(pack[0][4][:-1]) > 1 << 17:
            return None
        boxes = list(unpack)
        for src, offset, dst, dst_offset, extent, own, packed in pack:
            j = dst - 2 - 4 * i
            start, stop = [s.start for s in slices[i][j]], [s.stop for s in slices[i][j]]
            begin, end = start[p], stop[p]           # what is left for the tensor along dimension p
            for side, ghost in ((_LEFT_GHOST, left), (_RIGHT_GHOST, right)):
                if not present[p][side] or ghost[p].stop <= ghost[p].start:
                    continue
                if any(d != p and (a < g.start or b > g.stop) for d, (a, b, g) in enumerate(zip(start, stop, ghost))) or \
                        ghost[p].start < start[p] or ghost[p].stop > stop[p]:
                    return None
                part = list(extent)
                part[p] = ghost[p].stop - ghost[p].start
                held = hip_ops.contiguous_strides([int(g.stop) - int(g.start) for g in ghost])
                inside = sum((a - g.start) * s for d, (a, g, s) in enumerate(zip(start, ghost, held)) if d != p)
                boxes.append((2 + 4 * p + side, inside, dst, dst_offset + (ghost[p].start - start[p]) * packed[p], part, held, packed))
                begin, end = (ghost[p].stop, end) if side == _LEFT_GHOST else (begin, ghost[p].start)
            part = list(extent)
            part[p] = end - begin
            boxes.append((src, offset + (begin - start[p]) * own[p], dst, dst_offset + (begin - start[p]) * packed[p], part, own, packed))
        return boxes


def _plan(dims, slices, buffers, tensor, forward):
    cache = getattr(slices, "plans", None)
    present = tuple([b is not None for sides in buffers for b in sides])
    key = (dims, forward, tensor.shape, tensor.stride(), tensor.element_size(), present)
    plan = None if cache is None else cache.get(key)
    if plan is None:
        present = [[b is not None for b in sides] for sides in buffers]
        plan = _Plan(dims, slices, present, tuple(int(n) for n in tensor.shape), [int(s) for s in tensor.stride()],
                     tensor.element_size(), forward)
        if cache is not None:
            cache[key] = plan
    return plan


def _views(buffers, plan, tensor, bases):
    """The views of every dimension's four buffers; their addresses go into ``bases``."""
    out, dtype = [], tensor.dtype
    for sides, dim in zip(buffers, plan.dims):
        views = []
        for buffer, extent in zip(sides, dim[0]):
            if buffer is None:
                views.append(None)
                bases.append(0)
                continue
            view = buffer.get_view(extent)
            if view.dtype != dtype:
                raise ValueError(f"buffer {tuple(view.shape)}/{view.dtype} does not match a tensor of {dtype}")
            views.append(view)
            bases.append(view.data_ptr())
        hip_ops._require_gpu(*views)
        out.append(views)
    return out


def _before(plan, i, bases):
    """The launches ahead of the messages of dimension ``i``: the ghosts of the one before are unpacked, this one's strips
    packed.  One launch for both, unless a strip goes into a buffer that still holds a ghost."""
    if i == len(plan.dims):
        return [plan.dims[-1][2]] if plan.dims else []
    _, pack, _, both = plan.dims[i]
    if i == 0:
        return [pack]
    return [both] if both is not None and not _share(bases, i) else [plan.dims[i - 1][2], pack]


def _in_order(plan, bases):
    """All launches of a forward exchange that sends no messages."""
    return [plan.first] + [launch for i in range(len(plan.dims) + 1) for launch in _before(plan, i, bases)]


def _share(bases, i):
    """Is one of dimension ``i``'s bulk buffers a ghost buffer of dimension ``i - 1``?"""
    ghosts = {bases[4 * i - 2 + _LEFT_GHOST], bases[4 * i - 2 + _RIGHT_GHOST]} - {0}
    return bases[2 + 4 * i + _LEFT_BULK] in ghosts or bases[2 + 4 * i + _RIGHT_BULK] in ghosts


def _swap(P_x, neighbor_ranks_i, out_left, out_right, in_left, in_right):
    """Left message travels with tag 0, right message with tag 1; the receiver
    matches the opposite tag (reference :55-61)."""
    lrank, rrank = neighbor_ranks_i
    sends, recvs = [], []
    if in_left is not None and lrank != PROC_NULL:
        recvs.append((lrank, in_left, _RTAG))
    if in_right is not None and rrank != PROC_NULL:
        recvs.append((rrank, in_right, _LTAG))
    if out_left is not None and lrank != PROC_NULL:
        sends.append((lrank, out_left, _LTAG))
    if out_right is not None and rrank != PROC_NULL:
        sends.append((rrank, out_right, _RTAG))
    if sends or recvs:
        P_x._world.transport.exchange(P_x, sends, recvs)


def _adjoint(P_x, slices, buffers, neighbor_ranks, grad_output):
    """In place on the incoming gradient, as the reference (:98)."""
    if not grad_output.is_contiguous():
        raise ValueError("HaloExchange adjoint needs a contiguous gradient")

    hip_ops._require_gpu(grad_output)
    plan = _plan(P_x.dim, slices, buffers, grad_output, False)
    bases = [0, grad_output.data_ptr()]
    views = _views(buffers, plan, grad_output, bases)
    add_dtype = hip_ops._ADD_DTYPES.get(grad_output.dtype)
    if add_dtype is None and plan.adds:
        raise ValueError(f"accumulating unpack is not available for {grad_output.dtype}")
    for i in reversed(range(len(views))):
        lbb, lgb, rbb, rgb = views[i]
        _, out, clear, adds = plan.dims[i]
        out.run(bases, op=_lib.DDL_OP_COPY if clear else _lib.DDL_OP_MOVE)
        if clear:
            clear.zero(grad_output)
        _swap(P_x, neighbor_ranks[i], lgb, rgb, lbb, rbb)
        for launch in adds:
            launch.run(bases, op=_lib.DDL_OP_ADD, dtype=add_dtype)
    return grad_output


def native_exchange(input, P_x, slices, buffers, neighbor_ranks):
    """Forward and, if it requires gradients, adjoint for tensors like ``input`` as native moves, where no message is sent
    between their launches (the live rank of a solo transport).  None otherwise, and where the general way raises or clears
    ghosts in a launch of its own."""
    if not P_x.active or P_x.size == 1 or type(P_x._world.transport) is not SoloTransport or not input.is_cuda:
        return None
    epoch, bases = _lib.buffers_epoch(), [0, 0]
    adjoint = None
    try:
        plan = _plan(P_x.dim, slices, buffers, input, True)
        views = [v for sides in _views(buffers, plan, input, bases) for v in sides]
        if input.requires_grad:
            like = torch.empty(input.shape, dtype=input.dtype, device="meta")       # contiguous, as the result and its gradient are
            adjoint = _plan(P_x.dim, slices, buffers, like, False)
    except (RuntimeError, ValueError):
        return None
    forward = hip_ops.native_moves(epoch, input, tuple(input.shape),
                                   [(launch, _lib.DDL_OP_COPY, _lib.DDL_DT_BITS) for launch in _in_order(plan, bases)], views)
    if adjoint is None:
        return forward, None
    add_dtype = hip_ops._ADD_DTYPES.get(input.dtype)
    if add_dtype is None or any(clear for _, _, clear, _ in adjoint.dims):
        return None
    back = []
    for _, out, _, adds in reversed(adjoint.dims):
        back += [(out, _lib.DDL_OP_MOVE, _lib.DDL_DT_BITS)] + [(launch, _lib.DDL_OP_ADD, add_dtype) for launch in adds]
    return forward, hip_ops.native_moves(epoch, like, None, back, views,
                                         general=functools.partial(_adjoint, P_x, slices, buffers, neighbor_ranks))


class HaloExchangeFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, input, P_x, slices, buffers, neighbor_ranks):
        ctx.slices = slices
        ctx.buffers = buffers
        ctx.neighbor_ranks = neighbor_ranks
        ctx.P_x = P_x
        ctx.device = input.device

        if not P_x.active:
            return zero_volume_tensor(input.shape[0], device=input.device)
        if P_x.size == 1:
            return input

        # The reference works on a copy because marking the input dirty breaks
        # some downstream layers (halo_exchange.py:26-30); the copy runs on the
        # box kernel, which packs the first dimension's strips in the same launch.
        src = input.detach()
        hip_ops._require_gpu(src)
        output = torch.empty_like(src, memory_format=torch.contiguous_format)
        plan = _plan(P_x.dim, slices, buffers, src, True)
        bases = [src.data_ptr(), output.data_ptr()]
        views = _views(buffers, plan, output, bases)
        plan.first.run(bases)
        for i, (lbb, lgb, rbb, rgb) in enumerate(views):
            for launch in _before(plan, i, bases):
                launch.run(bases)
            _swap(P_x, neighbor_ranks[i], lbb, rbb, lgb, rgb)
        for launch in _before(plan, len(views), bases):
            launch.run(bases)
        return output

    @staticmethod
    def backward(ctx, grad_output):
        P_x, slices, buffers = ctx.P_x, ctx.slices, ctx.buffers
        if not P_x.active:
            return zero_volume_tensor(grad_output.shape[0], device=ctx.device), None, None, None, None
        if P_x.size == 1:
            return grad_output, None, None, None, None

        ctx.mark_dirty(grad_output)
        _adjoint(P_x, slices, buffers, ctx.neighbor_ranks, grad_output)
        return grad_output, None, None, None, None
