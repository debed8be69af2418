"""The layers' native autograd nodes against the torch.autograd.Functions behind them: the same bits, and what torch does around a
node (hooks on saved tensors, versions, a second pass, transforms, copies of layers) as before."""

import copy
import pickle
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NODES = ("linear_shard", "layer_norm_shard", "layer_norm_node", "embedding_shard", "move", "alias", "attachable", "unobserved")


class _WithoutNodes:

    def __init__(self, real):
        self.real = real

    def __getattr__(self, name):
        return (lambda *args: None) if name in NODES else getattr(self.real, name)


@pytest.fixture
def general(monkeypatch):
    """general(fn): fn() without the nodes."""
    from distdl_amd import _lib

    def run(fn):
        real = _lib.front()
        monkeypatch.setattr(_lib, "_front", _WithoutNodes(real))
        try:
            return fn()
        finally:
            monkeypatch.setattr(_lib, "_front", real)
    return run


def _randn(*shape, dtype=torch.float32, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed + sum(shape)), device="cuda").to(dtype)


def _partition(workers, shape, rank=0):
    from distdl_amd.backends.stub_hip import SimWorld
    world = SimWorld(workers)
    return world, world.partition(rank).create_partition_inclusive(list(range(workers))).create_cartesian_topology_partition(shape)


def _case(name):
    """(layer, input, parameters) of a small layer, buffers filled."""
    from distdl_amd import nn
    from distdl_amd.backends.stub_hip import BufferManager
    from distdl_amd.nn.layernorm import BWD_SUMS_TAG
    from distdl_amd.nn.layernorm import STATS_TAG
    manager = BufferManager()
    if name == "linear_ag":
        layer, x = nn.DistributedLinearAllGather(_partition(4, [1, 1, 4])[1], 72, 96, dtype=torch.bfloat16), _randn(2, 9, 72, dtype=torch.bfloat16)
    elif name == "linear":
        from distdl_amd.backends.stub_hip import SimWorld
        team = SimWorld(2).partition(0)
        P_x = team.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1])
        P_w = team.create_partition_inclusive([0, 1]).create_cartesian_topology_partition([2, 1])
        P_y = team.create_partition_inclusive([0, 1]).create_cartesian_topology_partition([1, 2])
        layer, x = nn.DistributedLinear(P_x, P_y, P_w, 31, 34), _randn(11, 31)
    elif name == "linear_rs":
        layer, x = nn.DistributedLinearReduceScatter(_partition(4, [1, 1, 4])[1], 64, 40, dtype=torch.bfloat16), _randn(2, 9, 16, dtype=torch.bfloat16)
    elif name in ("layernorm", "layernorm_narrow"):
        cols = 768 if name == "layernorm" else 163
        layer, x = nn.DistributedLayerNorm(_partition(1, [1, 1, 1])[1], [cols]), _randn(3, 17, cols)
    elif name == "layernorm_shared":
        world, P = _partition(4, [1, 1, 4])
        layer, x = nn.DistributedLayerNorm(P, [512]), _randn(3, 17, 128)
        peers = [torch.stack((0.1 * _randn(51, seed=q), 128 + _randn(51, seed=9 + q)), dim=1) for q in range(4)]
        sums = [_randn(51, 2, seed=q) for q in range(4)]
        world.transport.set_gather_provider(STATS_TAG, lambda P, t: list(peers), constant=True)
        world.transport.set_gather_provider(BWD_SUMS_TAG, lambda P, t: list(sums))
        with torch.no_grad():
            layer(x)
    elif name == "embedding":
        layer = nn.DistributedEmbedding(_partition(1, [1, 1, 1])[1], 50, 24, padding_idx=3)
        x = torch.arange(60, device="cuda").reshape(4, 15) % 37
    elif name == "repartition":
        world, P_x = _partition(3, [1, 3])
        P_y = world.partition(0).create_partition_inclusive([0, 1, 2]).create_cartesian_topology_partition([3, 1])
        world.transport.set_peer_shape_provider(lambda P, index, mine: [7, [6, 5, 5][int(index[1])]])
        layer, x = nn.Repartition(P_x, P_y, buffer_manager=manager), _randn(7, 6)
    elif name == "exchange":
        width = np.array([[0, 0], [0, 0], [1, 1], [1, 1]])
        layer, x = nn.HaloExchange(_partition(9, [1, 1, 3, 3], 4)[1], width, width, width, buffer_manager=manager), _randn(2, 3, 8, 9)
    elif name == "staging":
        class Staging(nn.DistributedFeatureConv2d):
            def forward(self, input):
                return self.stage_input(input)
        layer = Staging(_partition(4, [1, 1, 2, 2])[1], in_channels=3, out_channels=1, kernel_size=3, padding=1, bias=False, buffer_manager=manager)
        x = _randn(2, 3, 8, 9)
    with torch.no_grad():
        for k, p in enumerate(layer.parameters()):
            p.copy_(_randn(*p.shape, seed=k))
        layer(x)
    layer.__dict__["pooled"] = manager.buffers_map
    params = [] if name == "staging" else list(layer.parameters())
    return layer, x.requires_grad_(True) if x.is_floating_point() else x, params


CASES = ["linear_ag", "linear", "linear_rs", "layernorm", "layernorm_narrow", "layernorm_shared", "embedding", "repartition", "exchange", "staging"]
SAVING = CASES[:7]


def _fill(layer):
    """What the peers have sent; a pass leaves its own strips in the same buffers."""
    for pool in layer.__dict__["pooled"].values():
        for k, b in enumerate(pool):
            b.raw_buffer.copy_(_randn(b.raw_buffer.numel(), seed=k))


def _step(layer, x, wanted, dy, **kwargs):
    _fill(layer)
    y = layer(x)
    return [y, *torch.autograd.grad(y, wanted, dy.clone(), **kwargs)]


def _same(a, b):
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert p.shape == q.shape and p.dtype == q.dtype and p.stride() == q.stride() and p.requires_grad == q.requires_grad
        assert torch.equal(p.detach().contiguous().view(torch.uint8), q.detach().contiguous().view(torch.uint8))


@pytest.mark.parametrize("name", CASES)
def test_nodes_compute_what_the_functions_do(general, name):
    layer, x, params = _case(name)
    wanted = ([x] if x.is_floating_point() else []) + params
    dy = _randn(*layer(x).shape, dtype=params[0].dtype if params else x.dtype, seed=5)
    assert type(layer(x).grad_fn).__name__ != type(general(lambda: layer(x)).grad_fn).__name__
    _same(_step(layer, x, wanted, dy), general(lambda: _step(layer, x, wanted, dy)))
    for some in [[w] for w in wanted]:
        _same(_step(layer, x, some, dy), general(lambda: _step(layer, x, some, dy)))
    with torch.no_grad():
        for run in (lambda fn: fn(), general):
            _fill(layer)
            out = run(lambda: [layer(x)])
            with torch.enable_grad():
                _same(out, [_step(layer, x, wanted, dy)[0].detach()])
    _same(_step(layer, x, wanted, dy, create_graph=True), general(lambda: _step(layer, x, wanted, dy, create_graph=True)))
    if x.is_floating_point():
        turned = x.detach().transpose(0, 1).contiguous().transpose(0, 1).requires_grad_(True)
        _same(_step(layer, turned, [turned] + params, dy), general(lambda: _step(layer, turned, [turned] + params, dy)))
    # a gradient that the native adjoint does not take
    y, z = layer(x), general(lambda: layer(x))
    _fill(layer)
    odd = torch.empty(*dy.shape[:-1], dy.shape[-1] + 1, dtype=dy.dtype, device="cuda")[..., :-1].copy_(dy)
    if name == "exchange":
        for t in (y, z):
            with pytest.raises(ValueError, match="contiguous gradient"):
                torch.autograd.grad(t, wanted, odd)
    else:
        mine = torch.autograd.grad(y, wanted, odd)
        _fill(layer)
        _same(mine, general(lambda: torch.autograd.grad(z, wanted, odd)))


@pytest.mark.parametrize("name", SAVING)
def test_a_second_pass_hooks_on_saved_tensors_and_versions(general, name):
    layer, x, params = _case(name)
    wanted = ([x] if x.is_floating_point() else []) + params
    dy = _randn(*layer(x).shape, dtype=params[0].dtype, seed=5)
    y = layer(x)
    first = torch.autograd.grad(y, wanted, dy, retain_graph=True)
    _same(first, torch.autograd.grad(y, wanted, dy))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, wanted, dy)

    def hooked():
        packed = []

        def pack(t):
            packed.append((tuple(t.shape), t.dtype))
            return t.cpu()
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
            y = layer(x)
        return packed, torch.autograd.grad(y, wanted, dy)
    (mine, a), (theirs, b) = hooked(), general(hooked)
    assert [(int(np.prod(s)), t) for s, t in mine] == [(int(np.prod(s)), t) for s, t in theirs]
    _same(a, b)
    if x.is_floating_point():
        h = x * 1
        y = layer(h)
        with torch.no_grad():
            h.add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(y, params, dy)


@pytest.mark.parametrize("name", ["linear_ag", "layernorm", "repartition", "exchange", "staging"])
def test_transforms_and_tangents_see_the_functions(general, name):
    """The native nodes stay out of the way: what a transform or a tangent meets is what it meets without them."""
    layer, x, _ = _case(name)

    def outcome(fn):
        try:
            out = fn()
        except Exception as e:
            return type(e)
        return [tuple(t.shape) for t in out]

    def tangent():
        with torch.autograd.forward_ad.dual_level():
            y = layer(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
            return [t for t in torch.autograd.forward_ad.unpack_dual(y) if t is not None]
    for fn in (tangent, lambda: [torch.func.grad(lambda t: layer(t).float().sum())(x.detach())],
               lambda: [torch.func.vmap(layer)(torch.stack([x.detach(), x.detach()]))]):
        assert outcome(fn) == general(lambda: outcome(fn))


def test_what_layers_keep_can_be_copied():
    """Native objects stay with their layer: a copy of what holds them makes its own."""
    for name, kept in (("repartition", "_moves"), ("exchange", "_moves"), ("staging", "_moves"), ("layernorm", "_adjoint_calls"), ("linear_rs", None)):
        layer, x, _ = _case(name)
        layer(x)
        own = getattr(layer, kept) if kept else layer.reduce_scatter._adjoint
        assert own.value is not None and copy.deepcopy(own).value is None and pickle.loads(pickle.dumps(own)).value is None
    copy.deepcopy(_case("staging")[0]._staging_plan)


def test_moves_after_a_buffer_has_been_reallocated(general):
    """The pooled buffers grow between forward and adjoint: the adjoint moves through the new ones."""
    layer, x, _ = _case("repartition")
    manager, dy = layer.buffer_manager, _randn(*layer(x).shape, seed=5)

    def grow_between():
        _fill(layer)
        y = layer(x)
        pool = next(iter(manager.buffers_map.values()))
        for b in pool:
            b.expand(b.capacity + 8)
        for k, b in enumerate(pool):
            b.raw_buffer.fill_(k + 2.0)
        return [torch.autograd.grad(y, x, dy)[0], layer(x)]
    _same(grow_between(), general(grow_between))


def test_a_gather_that_raises_keeps_its_type():
    from distdl_amd.nn.layernorm import BWD_SUMS_TAG

    class Mine(Exception):
        pass

    def refuse(P, t):
        raise Mine("no")
    layer, x, _ = _case("layernorm_shared")
    layer.P_x._world.transport.set_gather_provider(BWD_SUMS_TAG, refuse)
    y = layer(x)
    with pytest.raises(Mine):
        y.backward(torch.ones_like(y))


def test_the_transport_is_asked_again_on_every_call(general):
    """Moves that a solo transport made do not run once another transport is in its place."""
    layer, x, _ = _case("exchange")
    layer(x)
    world, sent = layer.P_x._world, []
    solo = world.transport

    class Wire(type(solo)):
        def exchange(self, P, sends, recvs):
            sent.append(len(sends))
    world.transport = Wire(world)
    layer(x)
    assert sent == [2, 2]
    world.transport = solo
    layer(x)
    assert sent == [2, 2]


def test_passes_of_several_threads():
    layer, x, params = _case("layernorm")
    dy = _randn(*x.shape, seed=5)
    want, errors = _step(layer, x, [x] + params, dy), []

    def body():
        try:
            for _ in range(20):
                _same(_step(layer, x, [x] + params, dy), want)
        except Exception as e:      # noqa: B902
            errors.append(e)
    threads = [threading.Thread(target=body) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors


@pytest.mark.parametrize("name", CASES)
def test_compiled_autograd_runs_through_the_nodes(general, name):
    """The bits of an ordinary pass, under the compiled one as it is recorded, with other values, and for another layer alike."""
    from torch._dynamo import compiled_autograd
    for seed in (5, 6):
        layer, x, params = _case(name)
        wanted = ([x] if x.is_floating_point() else []) + params
        dy = _randn(*layer(x).shape, dtype=params[0].dtype if params else x.dtype, seed=seed)
        want = [_step(layer, x, wanted, k * dy) for k in (1, 2)] + [_step(layer, x, wanted[-1:], dy)]
        with compiled_autograd._enable(lambda graph: graph):
            got = [_step(layer, x, wanted, k * dy) for k in (1, 2)] + [_step(layer, x, wanted[-1:], dy)]
        for a, b in zip(got, want):
            _same(a, b)
        assert type(layer(x).grad_fn).__name__ != type(general(lambda: layer(x)).grad_fn).__name__


@pytest.mark.parametrize("name", ["repartition", "exchange", "staging"])
def test_when_moves_are_made(monkeypatch, name):
    """At once where a gradient is recorded, else when an input like the last one comes again; they give what the general way does."""
    from distdl_amd import hip_ops
    layer, x, _ = _case(name)
    made, real = [], hip_ops.native_moves
    monkeypatch.setattr(hip_ops, "native_moves", lambda *args, **kwargs: made.append(1) or real(*args, **kwargs))
    plain, outs, counts = x.detach(), [], []

    def call(t):
        _fill(layer)
        made.clear()
        outs.append(layer(t).detach())
        counts.append(len(made))
    with torch.no_grad():
        for t in (x, plain, x, plain, plain, plain):
            call(t)
        assert counts == [0, 0, 0, 0, 1, 0]
    for t in (x, x, plain, plain, x):
        call(t)
    assert counts[6:] == [2, 0, 0, 1, 2]           # forward and adjoint
    for out in outs:
        assert torch.equal(out, outs[0])
