"""Performance cases: one rank's share of the layers' work, as a program calls it.

A case names a layer, its sizes, element type and partition.  ``prepare`` builds
what such a program holds before a step (the layer with its parameters, the
input, the gradient that will arrive, what the absent peers contribute), ``run``
is one step through the layer: the forward alone where a program only infers,
the forward and the gradients of input and parameters where it trains.

One rank is live (the solo transport); where a layer needs what its peers send,
the receive buffers or gather providers are filled beforehand.
"""

import math

import numpy as np
import torch

from distdl_amd.backends.stub_hip import BufferManager
from distdl_amd.backends.stub_hip import SimWorld
from distdl_amd.nn import DistributedEmbedding
from distdl_amd.nn import DistributedFeatureConv2d
from distdl_amd.nn import DistributedFeatureConv3d
from distdl_amd.nn import DistributedLayerNorm
from distdl_amd.nn import DistributedLinear
from distdl_amd.nn import DistributedLinearAllGather
from distdl_amd.nn import DistributedLinearReduceScatter
from distdl_amd.nn import HaloExchange
from distdl_amd.nn import Repartition
from distdl_amd.nn.layernorm import BWD_SUMS_TAG
from distdl_amd.nn.layernorm import STATS_TAG

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
REDUCE_SCATTER_TAG = ("reduce_scatter", None)
REDUCE_SCATTER_ADJOINT_TAG = ("reduce_scatter_adjoint", None)


def listed():
    return [
        # Training step of a layer norm whose rows are split over four workers: the smallest of the repository's
        # benchmark configurations ([16,512,1024] over [1,1,4]); 8 MiB, so launches and host work count.
        {"name": "layernorm_split", "layer": "layernorm", "dtype": "f32", "batch": 16, "tokens": 512, "features": 1024, "workers": 4,
         "train": True},
        # Training step of a layer norm over whole rows of a wide transformer's hidden state (the activation of the
        # linear configuration, [4,2048,8192] bf16).
        {"name": "layernorm_wide", "layer": "layernorm", "dtype": "bf16", "batch": 4, "tokens": 2048, "features": 8192, "workers": 1,
         "train": True},
        # Training step of the vocabulary-sharded embedding of the benchmark's configuration: most ids miss.
        {"name": "embedding_vocab", "layer": "embedding", "dtype": "bf16", "batch": 32, "tokens": 4096, "vocab": 128256,
         "rows": 16032, "dim": 4096, "ids": "uniform", "train": True},
        # Training step of the embedding as the reference shards it (whole vocabulary, an eighth of the columns), token
        # ids as in text: the most frequent one is several percent of all.
        {"name": "embedding_dim", "layer": "embedding", "dtype": "f32", "batch": 8, "tokens": 1024, "vocab": 50304, "rows": 50304,
         "dim": 512, "ids": "zipf", "train": True},
        # One token for each of eight sequences through the benchmark's linear shard: a decode step.
        {"name": "linear_decode", "layer": "linear_ag", "dtype": "bf16", "batch": 8, "tokens": 1, "in": 8192, "out": 28672, "workers": 8,
         "train": False},
        # The benchmark's linear shard on whole sequences: a prefill (M 8192, N 3584, K 8192).
        {"name": "linear_prefill", "layer": "linear_ag", "dtype": "bf16", "batch": 4, "tokens": 2048, "in": 8192, "out": 28672, "workers": 8,
         "train": False},
        # Training step of the plain linear layer in its default type, sizes that fit no tile (M 777, N 333, K 1024).
        {"name": "linear_ragged", "layer": "linear", "dtype": "f32", "batch": 777, "tokens": 1, "in": 1024, "out": 666, "workers": 2,
         "train": True},
        # Training step of the row-parallel linear: shard product, sum of eight partial outputs, and the adjoint.
        {"name": "linear_row_parallel", "layer": "linear_rs", "dtype": "bf16", "batch": 4, "tokens": 256, "in": 8192, "out": 4096,
         "workers": 8, "train": True},
        # The headline repartition, [8,4096,8192] bf16 from rows to columns over eight workers, and its adjoint.
        {"name": "repartition_even", "layer": "repartition", "dtype": "bf16", "shape0": 8, "shape1": 4096, "shape2": 8192, "workers": 8,
         "train": True},
        # A repartition whose extents divide by nothing: odd rows, odd runs of 16-bit elements.
        {"name": "repartition_ragged", "layer": "repartition", "dtype": "bf16", "shape0": 5, "shape1": 1531, "shape2": 3077, "workers": 4,
         "train": True},
        # Input staging of the benchmark's 3-D convolution (pad, ghosts, send slabs; [1,32,128^3] fp32) and its adjoint.
        {"name": "staging_3d", "layer": "staging", "dtype": "f32", "batch": 1, "channels": 32, "edge": 128, "spatial": 3, "split": 2,
         "rank": 0, "kernel": 3, "train": True},
        # Halo exchange of an interior worker between 2-D convolutions, dimension by dimension, and its adjoint.
        {"name": "exchange_2d", "layer": "exchange", "dtype": "f32", "batch": 8, "channels": 64, "edge": 130, "spatial": 2, "split": 3,
         "rank": 4, "kernel": 3, "train": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _either(rng, n):
    """``n`` as it came, or the multiple of 64 next to it: sizes in use are mostly round ones."""
    return max(64, n // 64 * 64) if rng.random() < 0.5 else n


def draw(rng):
    layer = rng.choice(["layernorm", "embedding", "linear_ag", "linear_ag", "linear", "linear_rs", "repartition", "staging", "exchange"])
    if layer == "layernorm":
        workers = rng.choice([1, 1, 2, 4])
        features = _either(rng, _log_int(rng, 64 * workers, 12288))
        rows = _log_int(rng, 64, max(64, min(65536, (1 << 26) // features)))
        batch = rng.choice([1, 2, 3, 4])
        return {"layer": layer, "dtype": rng.choice(["f32", "bf16", "f16"]), "batch": batch, "tokens": max(1, rows // batch),
                "features": features, "workers": workers, "train": rng.random() < 0.75}
    if layer == "embedding":
        vocab = _log_int(rng, 1000, 131072)
        rows = vocab if rng.random() < 0.6 else max(1, vocab // 8)
        dim = _either(rng, _log_int(rng, 64, 4096))
        batch = rng.choice([1, 4, 8, 32])
        tokens = _log_int(rng, 16, max(16, min(4096, (1 << 28) // (dim * batch))))
        while rows * dim > 1 << 28:
            dim = max(64, dim // 2)
        return {"layer": layer, "dtype": rng.choice(["f32", "bf16"]), "batch": batch, "tokens": tokens, "vocab": vocab, "rows": rows,
                "dim": dim, "ids": rng.choice(["uniform", "zipf"]), "train": rng.random() < 0.75}
    if layer in ("linear_ag", "linear", "linear_rs"):
        workers = {"linear_ag": 8, "linear": 2, "linear_rs": 8}[layer]
        dtype = {"linear_ag": rng.choice(["bf16", "bf16", "f16"]), "linear": "f32", "linear_rs": rng.choice(["bf16", "f16"])}[layer]
        train = layer != "linear_ag" or rng.random() < 0.4
        batch = rng.choice([1, 2, 4, 8])
        rows = _log_int(rng, 1, 256) if not train and rng.random() < 0.6 else _log_int(rng, 64, 8192)
        n_in, n_out = _either(rng, _log_int(rng, 256, 8192)), _either(rng, _log_int(rng, 256, 16384))
        # no more than the benchmark's product in 16 bits, a tenth of it in 32
        limit = (4.8e11 if dtype != "f32" else 4.8e10) / (6 if train else 2) * workers
        while rows * n_in * n_out > limit:
            rows = max(1, rows // 2)
        return {"layer": layer, "dtype": dtype, "batch": batch, "tokens": max(1, rows // batch), "in": n_in, "out": n_out,
                "workers": workers, "train": train}
    if layer == "repartition":
        workers = rng.choice([2, 4, 8])
        shape1 = _either(rng, _log_int(rng, 128, 4096))
        shape2 = _either(rng, _log_int(rng, 128, 8192))
        return {"layer": layer, "dtype": rng.choice(["f32", "bf16"]), "shape0": rng.randint(1, 8), "shape1": shape1, "shape2": shape2,
                "workers": workers, "train": rng.random() < 0.75}
    spatial = rng.choice([2, 3])
    edge = _log_int(rng, 24, 512) if spatial == 2 else _log_int(rng, 16, 128)
    most = max(1, (1 << 26) // edge ** spatial)
    batch = min(rng.choice([1, 2, 4, 8]), most)
    channels = _log_int(rng, 1, max(1, min(64, most // batch)))
    split, rank = rng.choice([(2, 0), (3, 4 if spatial == 2 else 13)])
    return {"layer": layer, "dtype": rng.choice(["f32", "f32", "bf16"]), "batch": batch, "channels": channels, "edge": edge,
            "spatial": spatial, "split": split, "rank": rank, "kernel": rng.choice([3, 5]), "train": rng.random() < 0.75}


class _Staging2d(DistributedFeatureConv2d):
    """The part of the distributed convolution in front of the local one."""

    def forward(self, input):
        return self.stage_input(input)


class _Staging3d(DistributedFeatureConv3d):

    def forward(self, input):
        return self.stage_input(input)


def _partition(workers, shape, rank=0):
    world = SimWorld(workers)
    team = world.partition(rank).create_partition_inclusive(list(range(workers)))
    return world, team.create_cartesian_topology_partition(shape)


def _set_parameters(layer, gen, scale):
    """Parameters from the generator alone: weights around zero (a layer norm's around one)."""
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn(p.shape, generator=gen, device=p.device) * scale)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _fill_buffers(manager, gen):
    """What the peers have sent: every pooled buffer filled from the generator."""
    for pool in manager.buffers_map.values():
        for buf in pool:
            buf.raw_buffer.normal_(generator=gen)


def _local(extent, workers, index=0):
    return extent // workers + (1 if index < extent % workers else 0)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    layer_name, workers = case["layer"], case.get("workers", 1)
    state = {"train": case["train"]}
    if layer_name == "layernorm":
        world, P = _partition(workers, [1, 1, workers])
        layer = DistributedLayerNorm(P, [case["features"]], dtype=dtype)
        cols = _local(case["features"], workers)
        rows = case["batch"] * case["tokens"]
        with torch.no_grad():
            layer.weight.copy_(1 + 0.1 * torch.randn(layer.weight.shape, generator=gen, device="cuda"))
            layer.bias.copy_(0.1 * torch.randn(layer.bias.shape, generator=gen, device="cuda"))
        if workers > 1:
            # row means and sums of squared deviations of standard normal shards; row sums of the backward pass
            peers = [torch.stack((torch.randn(rows, generator=gen, device="cuda") / math.sqrt(cols),
                                  torch.full((rows,), float(cols), device="cuda")), dim=1) for _ in range(workers)]
            sums = [torch.randn(rows, 2, generator=gen, device="cuda") * math.sqrt(cols) for _ in range(workers)]
            world.transport.set_gather_provider(STATS_TAG, lambda P, t: list(peers), constant=True)
            world.transport.set_gather_provider(BWD_SUMS_TAG, lambda P, t: list(sums))
        x = _randn(gen, (case["batch"], case["tokens"], cols), dtype)
        state["dy"] = _randn(gen, x.shape, dtype)
        state["wanted"] = [x, layer.weight, layer.bias]
    elif layer_name == "embedding":
        _, P = _partition(1, [1, 1, 1])
        layer = DistributedEmbedding(P, case["vocab"], case["dim"], dtype=dtype, vocab_shard=(0, case["rows"]))
        _set_parameters(layer, gen, 0.02)
        shape = (case["batch"], case["tokens"])
        if case["ids"] == "zipf":
            u = torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64)
            x = (torch.exp(u * math.log(case["vocab"] + 1)).long() - 1).clamp_(0, case["vocab"] - 1)
        else:
            x = torch.randint(0, case["vocab"], shape, generator=gen, device="cuda")
        state["dy"] = _randn(gen, shape + (case["dim"],), dtype) if case["train"] else None
        state["wanted"] = [layer.weight]
    elif layer_name == "linear_ag":
        _, P = _partition(workers, [1, 1, workers])
        layer = DistributedLinearAllGather(P, case["in"], case["out"], dtype=dtype)
        _set_parameters(layer, gen, 0.02)
        x = _randn(gen, (case["batch"], case["tokens"], case["in"]), dtype)
        state["dy"] = _randn(gen, (case["batch"], case["tokens"], _local(case["out"], workers)), dtype) if case["train"] else None
        state["wanted"] = [x, layer.weight, layer.bias]
    elif layer_name == "linear":
        world = SimWorld(workers)
        team = world.partition(0)
        P_x = team.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1])
        P_w = team.create_partition_inclusive(list(range(workers))).create_cartesian_topology_partition([workers, 1])
        P_y = team.create_partition_inclusive(list(range(workers))).create_cartesian_topology_partition([1, workers])
        layer = DistributedLinear(P_x, P_y, P_w, case["in"], case["out"]).to(dtype)
        _set_parameters(layer, gen, 0.02)
        x = _randn(gen, (case["batch"] * case["tokens"], case["in"]), dtype)
        state["dy"] = _randn(gen, (x.shape[0], _local(case["out"], workers)), dtype)
        state["wanted"] = [x, layer.sublinear.weight, layer.sublinear.bias]
    elif layer_name == "linear_rs":
        world, P = _partition(workers, [1, 1, workers])
        layer = DistributedLinearReduceScatter(P, case["in"], case["out"], dtype=dtype)
        _set_parameters(layer, gen, 0.02)
        x = _randn(gen, (case["batch"], case["tokens"], _local(case["in"], workers)), dtype)
        partial = [_randn(gen, (case["batch"], case["tokens"], case["out"]), dtype) for _ in range(workers)]
        pieces = [_randn(gen, (case["batch"], case["tokens"], _local(case["out"], workers, r)), dtype) for r in range(workers)]
        world.transport.set_gather_provider(REDUCE_SCATTER_TAG, lambda P, t: list(partial))
        world.transport.set_gather_provider(REDUCE_SCATTER_ADJOINT_TAG, lambda P, t: list(pieces))
        state["dy"] = _randn(gen, (case["batch"], case["tokens"], _local(case["out"], workers)), dtype)
        state["wanted"] = [x, layer.weight, layer.bias]
    elif layer_name == "repartition":
        world, P_x = _partition(workers, [1, workers, 1])
        P_y = world.partition(0).create_partition_inclusive(list(range(workers))).create_cartesian_topology_partition([1, 1, workers])
        world.transport.set_peer_shape_provider(
            lambda P, index, mine: [case["shape0"], _local(case["shape1"], workers, int(index[1])), case["shape2"]])
        manager = BufferManager()
        layer = Repartition(P_x, P_y, buffer_manager=manager)
        x = _randn(gen, (case["shape0"], _local(case["shape1"], workers), case["shape2"]), dtype)
        with torch.no_grad():
            state["dy"] = _randn(gen, layer(x).shape, dtype)
        _fill_buffers(manager, gen)
        state["wanted"] = [x]
    else:
        spatial, split, kernel = case["spatial"], case["split"], case["kernel"]
        _, P = _partition(split ** spatial, [1, 1] + [split] * spatial, case["rank"])
        manager = BufferManager()
        shape = (case["batch"], case["channels"]) + (case["edge"],) * spatial
        if layer_name == "staging":
            kind = _Staging2d if spatial == 2 else _Staging3d
            layer = kind(P, in_channels=case["channels"], out_channels=1, kernel_size=kernel, padding=kernel // 2, bias=False,
                         buffer_manager=manager)
        else:
            # a worker at index i receives a ghost strip from each neighbour it has, and sends it as much
            width = np.zeros((2 + spatial, 2), dtype=int)
            width[2:, 0] = kernel // 2 if case["rank"] else 0
            width[2:, 1] = kernel // 2
            layer = HaloExchange(P, width, width, width, buffer_manager=manager)
        x = _randn(gen, shape, dtype)
        with torch.no_grad():
            state["dy"] = _randn(gen, layer(x).shape, dtype)
        _fill_buffers(manager, gen)
        # the exchange's adjoint works in place on the gradient it is handed, in a network the fresh result of the layer
        # behind it; each step hands over a copy
        state["fresh"] = layer_name == "exchange"
        state["wanted"] = [x]
    if case["train"] and x.is_floating_point():
        x.requires_grad_(True)
    state["layer"], state["x"] = layer, x
    return state


def run(state):
    layer, x = state["layer"], state["x"]
    if not state["train"]:
        with torch.no_grad():
            return layer(x)
    dy = state["dy"].clone() if state.get("fresh") else state["dy"]
    y = layer(x)
    return [y, *torch.autograd.grad(y, state["wanted"], dy)]


def work(case):
    """Inputs read once, outputs written once."""
    es, train, workers = SIZE[case["dtype"]], case["train"], case.get("workers", 1)
    layer = case["layer"]
    rows = case.get("batch", 1) * case.get("tokens", 1)
    if layer == "layernorm":
        cols = _local(case["features"], workers)
        # x and y; dy and dx; parameters and their gradients; the peers' pairs of row sums
        nbytes = rows * cols * es * (4 if train else 2) + cols * es * (4 if train else 2)
        if workers > 1:
            nbytes += rows * 8 * workers * (2 if train else 1)
        return {"bytes": nbytes, "flops": rows * cols * (20 if train else 8)}
    if layer == "embedding":
        hit = rows * case["rows"] / case["vocab"]
        if case["ids"] == "zipf":
            hit = rows * math.log(case["rows"] + 1) / math.log(case["vocab"] + 1)
        row_bytes = case["dim"] * es
        distinct = min(hit, case["rows"] * (1 - math.exp(-hit / case["rows"])))
        nbytes = rows * 8 + distinct * row_bytes + rows * row_bytes
        if train:
            nbytes += hit * row_bytes + case["rows"] * row_bytes
        return {"bytes": nbytes, "flops": hit * case["dim"] if train else 0}
    if layer in ("linear_ag", "linear", "linear_rs"):
        n_in = _local(case["in"], workers) if layer == "linear_rs" else case["in"]
        n_out = case["out"] if layer == "linear_rs" else _local(case["out"], workers)
        x, w, y = rows * n_in, n_in * n_out + n_out, rows * n_out
        elements = x + w + y + ((y + x + w) if train else 0)
        if layer == "linear_rs":
            # this worker's slab of every peer's partial output and the slab it keeps; the peers' gradient pieces and its own
            elements = 2 * (x + w + y)
        return {"bytes": elements * es, "flops": (6 if train else 2) * rows * n_in * n_out}
    if layer == "repartition":
        shard = case["shape0"] * _local(case["shape1"], workers) * case["shape2"]
        out = case["shape0"] * case["shape1"] * _local(case["shape2"], workers)
        # a shard packed (read and written), the received boxes unpacked (read and written); the adjoint as much again
        return {"bytes": 2 * (shard + out) * es * (2 if train else 1), "flops": 0}
    spatial, half = case["spatial"], case["kernel"] // 2
    planes, edge = case["batch"] * case["channels"], case["edge"]
    sides = 2 if case["rank"] else 1
    face = planes * edge ** (spatial - 1) * half * sides * spatial
    if layer == "staging":
        # on a rank at the corner of the domain the other sides are zero padding
        shard, padded = planes * edge ** spatial, planes * (edge + 2 * half) ** spatial
        return {"bytes": (shard + padded + 2 * face + (2 * shard if train else 0)) * es, "flops": 0}
    whole = planes * edge ** spatial
    return {"bytes": (2 * whole + 2 * face + ((2 * whole + 2 * face) if train else 0)) * es, "flops": 0}


# Four times the relative error of these paths against the same sums in 64 bits (1.3e-6 for the longest fp32 products,
# one rounding of the result in the 16-bit types: 1.7e-3 and 2.2e-4).
RELATIVE = {"f32": 5e-6, "bf16": 7e-3, "f16": 1e-3}


def tolerance(case):
    """Moves keep every bit (the exchange's adjoint adds, in the order of the dimensions)."""
    if case["layer"] in ("repartition", "staging", "exchange") or (case["layer"] == "embedding" and not case["train"]):
        return "exact"
    return {"rel": RELATIVE[case["dtype"]]}
