"""GPU parity of the shard-compute kernels (LayerNorm, Embedding, Linear) and of
the layers wrapping them, through the C ABI.

Tolerances (from the task statement of this build): LayerNorm fp32 within 1e-5
relative, Linear bf16 within 2e-2 relative, Embedding bit-exact.  "Relative" is
taken with respect to the magnitude of the exact (fp64 oracle) result, with an
absolute floor of the same size because normalised outputs cross zero."""

import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import embedding as o_emb
from oracle import layernorm as o_ln
from oracle import linear as o_lin
from oracle import repartition as o_rep

pytestmark = pytest.mark.gpu

LN_RTOL = 1e-5
LIN_RTOL = 2e-2


@pytest.fixture(scope="module")
def ops():
    import distdl_amd  # noqa: F401
    from distdl_amd import hip_ops
    return hip_ops


def bits16(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


# ---------------------------------------------------------------- LayerNorm --

def _ln_case(ops, shards_cpu, gamma_full, beta_full, eps, live=0, strict=True):
    """Runs the two kernels for worker ``live`` of the reduction group; the
    other workers' partial statistics come from the oracle (fp64 -> fp32)."""
    cols = [s.shape[-1] for s in shards_cpu]
    x = torch.from_numpy(shards_cpu[live]).cuda()
    x2d = x.reshape(-1, cols[live])
    stats = ops.ln_partial_stats(x2d)
    want_stats = o_ln.partial_stats(shards_cpu[live])
    got_stats = stats.cpu().numpy().astype(np.float64)
    scale = np.abs(shards_cpu[live]).max()
    assert np.allclose(got_stats[:, 0], want_stats[:, 0], rtol=LN_RTOL, atol=LN_RTOL * scale)
    assert np.allclose(got_stats[:, 1], want_stats[:, 1], rtol=LN_RTOL, atol=LN_RTOL * scale * scale * cols[live])
    parts = []
    for p, s in enumerate(shards_cpu):
        parts.append(stats if p == live else torch.from_numpy(o_ln.partial_stats(s).astype(np.float32)).cuda())
    gathered = torch.stack(parts).contiguous()
    offs = np.cumsum([0] + cols)
    g = None if gamma_full is None else torch.from_numpy(gamma_full[offs[live]:offs[live + 1]].copy()).cuda()
    b = None if beta_full is None else torch.from_numpy(beta_full[offs[live]:offs[live + 1]].copy()).cuda()
    y, mean, rstd = ops.ln_normalize_affine(x2d, gathered, cols, g, b, eps, want_stats=True)
    torch.cuda.synchronize()
    _ln_joined_equals_two_launches(ops, x2d, gathered, live, cols, g, b, eps, y, mean, rstd)
    gs = [None if gamma_full is None else gamma_full[offs[p]:offs[p + 1]] for p in range(len(cols))]
    bs = [None if beta_full is None else beta_full[offs[p]:offs[p + 1]] for p in range(len(cols))]
    exact = o_ln.forward_shards(shards_cpu, gs, bs, eps, dtype=np.float64)[live].reshape(-1, cols[live])
    ref32 = o_ln.forward_shards(shards_cpu, gs, bs, eps, dtype=np.float32)[live].reshape(-1, cols[live])
    got = y.cpu().numpy().astype(np.float64)
    if strict:
        bound = LN_RTOL * np.maximum(np.abs(exact), 1.0)
        assert (np.abs(got - exact) <= bound).all(), float(np.abs(got - exact).max())
    # and no worse than the reference's own fp32 op sequence
    assert np.abs(got - exact).max() <= max(4 * np.abs(ref32 - exact).max(), 3e-6)
    return got, exact


def _ln_joined_equals_two_launches(ops, x2d, gathered, live, cols, g, b, eps, y, mean=None, rstd=None):
    """The single launch that writes this worker's statistics and consumes the
    peers' (already in the table) gives the bits of the two launches: y, the
    combined mean and rstd, and the worker's own slot of the table."""
    if not ops.ln_joined_supported(x2d, len(cols), g, b):
        with pytest.raises(RuntimeError, match="code -5"):      # DDL_E_UNSUPP
            ops.ln_stats_normalize(x2d, gathered.clone(), live, cols, g, b, eps)
        return
    table = gathered.clone()
    table[live] = float("nan")          # the launch must produce this slot itself
    y2, mean2, rstd2 = ops.ln_stats_normalize(x2d, table, live, cols, g, b, eps, want_stats=True)
    torch.cuda.synchronize()
    assert torch.equal(table, gathered)
    assert torch.equal(y2.view(torch.uint8), y.view(torch.uint8))
    if mean is not None:
        assert torch.equal(mean2, mean) and torch.equal(rstd2, rstd)


def test_layernorm_config1_rank0(ops):
    """Global [16,512,1024] fp32 split 4-way along the features; rank 0 holds
    [16,512,256].  gamma = 1 + 0.1 N(0,1), beta = 0.1 N(0,1), eps = 1e-5."""
    gen = torch.Generator().manual_seed(1001)
    x = torch.randn(16, 512, 1024, generator=gen).numpy()
    gamma = (1 + 0.1 * torch.randn(1024, generator=gen)).numpy()
    beta = (0.1 * torch.randn(1024, generator=gen)).numpy()
    shards = [np.ascontiguousarray(x[..., 256 * p:256 * (p + 1)]) for p in range(4)]
    got, exact = _ln_case(ops, shards, gamma, beta, 1e-5)
    # the reference's own check: equal to torch layer_norm of the whole row (tests/layers/test_layernorm.py:185-263)
    want = F.layer_norm(torch.from_numpy(x), (1024,), torch.from_numpy(gamma), torch.from_numpy(beta), 1e-5)
    assert np.allclose(got, want[..., :256].reshape(-1, 256).numpy(), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols,pad", [(3, 0), (5, 0), (257, 0), (513, 1), (1021, 0), (1025, 0), (1027, 2), (2051, 0), (4097, 0), (8191, 1), (16383, 0), (16391, 0), (1024, 0), (4096, 4)])
def test_layernorm_in_place_through_the_c_abi(ops, dtype, cols, pad):
    """y written over x, dx over dy and over x, at lengths where a row's last piece starts on elements of the one in front of
    it -- in the same lane's next request, another lane's, another wavefront's -- and at aligned ones.  The results are
    those in memory of its own, but for a product and a sum that may be rounded together or one by one."""
    from distdl_amd import _lib
    lib, rows, stream = _lib.load(), 37, torch.cuda.current_stream().cuda_stream
    dt, pitch = ops._LN_DTYPES[dtype], cols + pad
    gen = torch.Generator(device="cuda").manual_seed(cols)
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    x, dy = rnd(rows, pitch).to(dtype), rnd(rows, pitch).to(dtype)
    gamma, beta = (1 + 0.1 * rnd(cols)).to(dtype), (0.1 * rnd(cols)).to(dtype)
    stats = torch.stack((0.1 * rnd(1, rows), cols * (1 + 0.1 * rnd(1, rows).abs())), dim=2).contiguous()
    sums, mean, rstd = rnd(1, rows, 2), torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
    work, widths = torch.empty(2 * 256 * cols, device="cuda"), _lib.i64_array([cols])
    p = lambda t: t.data_ptr()

    def normalize(src, dst):
        return lib.ddl_ln_normalize_affine(p(src), dt, rows, cols, pitch, p(stats), 1, widths, p(gamma), p(beta), 1e-5, p(dst), pitch, p(mean), p(rstd), stream)

    def whole(src, dst):
        return lib.ddl_layer_norm(p(src), dt, rows, cols, pitch, p(gamma), p(beta), 1e-5, p(dst), pitch, p(mean), p(rstd), stream)

    def dx(dy, x, dst):
        return lib.ddl_ln_bwd_input(p(dy), p(x), dt, rows, cols, pitch, pitch, p(mean), p(rstd), p(gamma), p(sums), 1, 1.0 / cols, p(dst), pitch, stream)

    def dx_params(dy, x, dst):
        dg, db, scratch = torch.empty(cols, dtype=dtype, device="cuda"), torch.empty(cols, dtype=dtype, device="cuda"), torch.empty(rows, 2, device="cuda")
        rc = lib.ddl_ln_bwd_partial_params(p(dy), p(x), dt, rows, cols, pitch, pitch, p(mean), p(rstd), p(gamma), p(scratch), p(work), work.numel(), stream)
        return rc or lib.ddl_ln_bwd_input_params(p(dy), p(x), dt, rows, cols, pitch, pitch, p(mean), p(rstd), p(gamma), p(sums), 1, 1.0 / cols, p(dst), pitch,
                                                 p(work), work.numel(), p(dg), p(db), stream)

    def dx_whole(dy, x, dst):
        dg, db = torch.empty(cols, dtype=dtype, device="cuda"), torch.empty(cols, dtype=dtype, device="cuda")
        return lib.ddl_ln_bwd_whole_rows(p(dy), p(x), dt, rows, cols, pitch, pitch, p(mean), p(rstd), p(gamma), 1.0 / cols, p(dst), pitch, p(work), work.numel(),
                                         p(dg), p(db), stream)
    one = {torch.float32: 2.0 ** -22, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]

    def same(got, want):
        got, want = got[:, :cols].double(), want[:, :cols].double()
        assert bool(((got - want).abs() <= one * (want.abs() + 8)).all()) if dtype == torch.float32 else bool(((got - want).abs() <= one * want.abs() + 2.0 ** -21).all())
    for call in (normalize, whole):
        apart, here = torch.full_like(x, 77), x.clone()
        _lib.check(call(x, apart), "out of place")
        _lib.check(call(here, here), "in place")
        same(here, apart)
        assert torch.equal(here[:, cols:], x[:, cols:])
    for call in [dx, dx_params] + ([dx_whole] if 512 < cols <= 8192 else []):
        apart = torch.full_like(x, 77)
        _lib.check(call(dy, x, apart), "out of place")
        for over in "dy", "x":
            here = (dy if over == "dy" else x).clone()
            _lib.check(call(here, x, here) if over == "dy" else call(dy, here, here), "in place")
            same(here, apart)


@pytest.mark.parametrize("cols", [[4, 4], [64, 64, 64], [300, 212], [1000, 24], [2048], [7, 9], [4100, 4100],
                                  [20000, 100], [8] * 70, [4] * 200, [2052, 4096], [8192, 16384], [16388, 12000],
                                  [4101, 33]])
@pytest.mark.parametrize("affine", [True, False])
def test_layernorm_shapes_and_paths(ops, cols, affine):
    """Wavefront rows (aligned, <= 2048 columns), workgroup rows (aligned, <=
    16384 columns), streamed rows (longer, with and without four-element
    accesses), unequal widths, more workers per row than a wavefront has lanes."""
    rng = np.random.default_rng(sum(cols))
    rows = 37
    shards = [(rng.standard_normal((rows, c)) * 3 + 1.5).astype(np.float32) for c in cols]
    total = sum(cols)
    gamma = (1 + 0.1 * rng.standard_normal(total)).astype(np.float32) if affine else None
    beta = (0.1 * rng.standard_normal(total)).astype(np.float32) if affine else None
    for live in {0, len(cols) - 1}:
        _ln_case(ops, shards, gamma, beta, 1e-5, live=live)


@pytest.mark.parametrize("cols", [1, 7, 64, 256, 300, 1024, 2048, 2052, 4096, 8192, 12000, 16384, 16388, 40001])
@pytest.mark.parametrize("affine", [True, False])
def test_layer_norm_single_launch_fp32(ops, cols, affine):
    """Rows held whole by one worker: one kernel, against torch's layer_norm in
    float64 (the call the reference makes in that branch, nn/layernorm.py:319)
    and against the oracle with a single shard."""
    rng = np.random.default_rng(cols)
    rows = 29
    x = (rng.standard_normal((rows, cols)) * 2 - 0.7).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32) if affine else None
    beta = (0.1 * rng.standard_normal(cols)).astype(np.float32) if affine else None
    g = None if gamma is None else torch.from_numpy(gamma).cuda()
    b = None if beta is None else torch.from_numpy(beta).cuda()
    y, mean, rstd = ops.layer_norm(torch.from_numpy(x).cuda(), g, b, 1e-5, want_stats=True)
    torch.cuda.synchronize()
    exact = F.layer_norm(torch.from_numpy(x).double(), (cols,), None if gamma is None else torch.from_numpy(gamma).double(),
                         None if beta is None else torch.from_numpy(beta).double(), 1e-5).numpy()
    oracle = o_ln.forward_shards([x], [gamma], [beta], 1e-5, dtype=np.float64)[0]
    assert np.allclose(oracle, exact, rtol=1e-12, atol=1e-12)
    got = y.cpu().numpy().astype(np.float64)
    assert (np.abs(got - exact) <= LN_RTOL * np.maximum(np.abs(exact), 1.0)).all(), float(np.abs(got - exact).max())
    m = x.astype(np.float64).mean(axis=1)
    v = x.astype(np.float64).var(axis=1)
    assert np.allclose(mean.cpu().numpy(), m, rtol=1e-5, atol=1e-5)
    assert np.allclose(rstd.cpu().numpy(), 1 / np.sqrt(v + 1e-5), rtol=1e-5)
    # a strided view (row pitch larger than the row) gives the same bits
    wide = torch.zeros(rows, cols + 8, device="cuda")
    wide[:, :cols] = torch.from_numpy(x).cuda()
    y2 = ops.layer_norm(wide[:, :cols], g, b, 1e-5)
    assert torch.equal(y2, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols", [[8], [256], [300], [2048], [6000], [20000], [256, 256, 256, 256], [300, 212], [4100, 4100]])
def test_layernorm_16_bit_elements(ops, dtype, cols):
    """bf16 / fp16 inputs, parameters and outputs with fp32 sums: one rounding
    of the exact result of the reference's op sequence on the same 16-bit
    inputs (2e-2 relative is the bar for bf16; these stay within 2^-7)."""
    rng = np.random.default_rng(sum(cols) + len(cols))
    rows = 21
    shards_t = [torch.from_numpy((rng.standard_normal((rows, c)) * 2 + 0.5).astype(np.float32)).to(dtype) for c in cols]
    total = sum(cols)
    gamma_t = torch.from_numpy((1 + 0.1 * rng.standard_normal(total)).astype(np.float32)).to(dtype)
    beta_t = torch.from_numpy((0.1 * rng.standard_normal(total)).astype(np.float32)).to(dtype)
    shards64 = [t.double().numpy() for t in shards_t]
    offs = np.cumsum([0] + cols)
    gs = [gamma_t.double().numpy()[offs[p]:offs[p + 1]] for p in range(len(cols))]
    bs = [beta_t.double().numpy()[offs[p]:offs[p + 1]] for p in range(len(cols))]
    exact = o_ln.forward_shards(shards64, gs, bs, 1e-5, dtype=np.float64)
    tol = 2.0 ** -7
    for live in {0, len(cols) - 1}:
        x2d = shards_t[live].cuda()
        g = gamma_t[offs[live]:offs[live + 1]].contiguous().cuda()
        b = beta_t[offs[live]:offs[live + 1]].contiguous().cuda()
        if len(cols) == 1:
            y = ops.layer_norm(x2d, g, b, 1e-5)
        else:
            stats = ops.ln_partial_stats(x2d)
            want_stats = o_ln.partial_stats(shards64[live])
            assert np.allclose(stats.cpu().numpy()[:, 0], want_stats[:, 0], rtol=1e-5, atol=1e-5)
            parts = [stats if p == live else torch.from_numpy(o_ln.partial_stats(shards64[p]).astype(np.float32)).cuda()
                     for p in range(len(cols))]
            gathered = torch.stack(parts).contiguous()
            y = ops.ln_normalize_affine(x2d, gathered, cols, g, b, 1e-5)
            _ln_joined_equals_two_launches(ops, x2d, gathered, live, cols, g, b, 1e-5, y)
        assert y.dtype == dtype
        got = y.cpu().double().numpy()
        assert (np.abs(got - exact[live]) <= tol * np.maximum(np.abs(exact[live]), 1.0)).all()


def test_layernorm_layer_takes_one_launch_once_the_peers_are_seeded(ops):
    """One live rank of four: the first forward runs stats, gather, normalize
    and leaves the peers' statistics in the layer's table; from then on the
    transport reports them as present beforehand and the layer needs a single
    launch.  Both give the oracle's result; the gradient path does the same."""
    from distdl_amd import _lib
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    from distdl_amd.nn.layernorm import STATS_TAG
    world = SimWorld(4)
    P_x = world.partition(0).create_partition_inclusive(list(range(4))).create_cartesian_topology_partition([1, 1, 4])
    layer = DistributedLayerNorm(P_x, [512])
    gen = torch.Generator().manual_seed(77)
    whole = torch.randn(3, 50, 512, generator=gen)
    shards = [np.ascontiguousarray(whole[..., 128 * p:128 * (p + 1)].numpy()) for p in range(4)]
    peers = [None] + [torch.from_numpy(o_ln.partial_stats(shards[p]).astype(np.float32)).cuda() for p in range(1, 4)]
    world.transport.set_gather_provider(STATS_TAG, lambda P, t: list(peers), constant=True)
    with torch.no_grad():
        layer.weight.copy_((1 + 0.1 * torch.randn(128, generator=gen)).view(1, 1, 128))
        layer.bias.copy_((0.1 * torch.randn(128, generator=gen)).view(1, 1, 128))
    gs = [layer.weight.detach().cpu().numpy().reshape(-1)] + [None] * 3
    bs = [layer.bias.detach().cpu().numpy().reshape(-1)] + [None] * 3
    exact = o_ln.forward_shards(shards, gs, bs, 1e-5, dtype=np.float64)[0]
    x = torch.from_numpy(shards[0]).cuda()
    lib = _lib.load()
    calls = []
    real = lib.ddl_ln_stats_normalize

    class Spy:
        def __getattr__(self, name):
            if name == "ddl_ln_stats_normalize":
                def counted(*args):
                    calls.append(name)
                    return real(*args)
                return counted
            return getattr(lib, name)
    saved = _lib.load
    _lib.load = lambda: Spy()
    try:
        layer._call_plan = None
        with torch.no_grad():
            y_first = layer(x)
            assert calls == []
            y_second = layer(x)
            assert calls == ["ddl_ln_stats_normalize"]
        xg = x.clone().requires_grad_(True)
        y_grad = layer(xg)
        assert len(calls) == 2
    finally:
        _lib.load = saved
        layer._call_plan = None
    torch.cuda.synchronize()
    for y in (y_first, y_second, y_grad.detach()):
        got = y.cpu().numpy().astype(np.float64)
        assert (np.abs(got - exact) <= LN_RTOL * np.maximum(np.abs(exact), 1.0)).all()
    assert torch.equal(y_first, y_second) and torch.equal(y_first, y_grad.detach())


def test_layernorm_layer_solo_without_a_provider_is_consistent(ops):
    """One live worker of four and nobody speaking for the others: the absent
    workers hold what the live one holds, in the forward's gather and in the
    backward's alike, so the layer is the layer norm of the live shard over its
    own columns and its gradients are that function's (torch autograd)."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    world = SimWorld(4)
    P_x = world.partition(0).create_partition_inclusive(list(range(4))).create_cartesian_topology_partition([1, 1, 4])
    layer = DistributedLayerNorm(P_x, [1024])
    gen = torch.Generator().manual_seed(151)
    with torch.no_grad():
        layer.weight.copy_((1 + 0.1 * torch.randn(layer.weight.shape, generator=gen)).cuda())
        layer.bias.copy_((0.1 * torch.randn(layer.bias.shape, generator=gen)).cuda())
    x = torch.randn(3, 37, 256, generator=gen)
    dy = torch.randn(3, 37, 256, generator=gen)
    for _ in range(2):                                  # the second call finds the statistics buffer of the first
        xg = x.cuda().requires_grad_(True)
        y = layer(xg)
        y.backward(dy.cuda())
        xr = x.double().requires_grad_(True)
        w = layer.weight.detach().cpu().double().reshape(-1).requires_grad_(True)
        b = layer.bias.detach().cpu().double().reshape(-1).requires_grad_(True)
        yr = F.layer_norm(xr, (256,), w, b, layer.eps)
        yr.backward(dy.double())
        assert torch.allclose(y.detach().cpu().double(), yr.detach(), rtol=1e-5, atol=1e-5)
        assert torch.allclose(xg.grad.cpu().double(), xr.grad, rtol=1e-4, atol=1e-5)
        assert torch.allclose(layer.weight.grad.cpu().double().reshape(-1), w.grad, rtol=1e-4, atol=1e-4)
        assert torch.allclose(layer.bias.grad.cpu().double().reshape(-1), b.grad, rtol=1e-4, atol=1e-4)
        layer.weight.grad = layer.bias.grad = None
        with torch.no_grad():
            y2 = layer(x.cuda())                        # the path without autograd: the same numbers
        assert torch.equal(y2, y.detach())


def test_layernorm_layer_single_worker_and_bf16(ops):
    """The layer on one worker takes the single-launch kernel (the reference's
    F.layer_norm branch) and is differentiable; a bf16 forward beside it."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    torch.manual_seed(3)
    x = torch.randn(6, 10, 96)
    ref = torch.nn.LayerNorm(96)
    with torch.no_grad():
        ref.weight.copy_(1 + 0.1 * torch.randn(96))
        ref.bias.copy_(0.1 * torch.randn(96))

    def body(P_world):
        P_x = P_world.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1, 1])
        layer = DistributedLayerNorm(P_x, 96)
        with torch.no_grad():
            layer.weight.copy_(ref.weight.reshape(1, 1, 96))
            layer.bias.copy_(ref.bias.reshape(1, 1, 96))
        xg = x.cuda().requires_grad_(True)
        y = layer(xg)
        y.backward(torch.ones_like(y) * 0.5 + y.detach())
        half = DistributedLayerNorm(P_x, 96, dtype=torch.bfloat16)
        with torch.no_grad():
            half.weight.copy_(ref.weight.reshape(1, 1, 96))
            half.bias.copy_(ref.bias.reshape(1, 1, 96))
            yh = half(x.cuda().to(torch.bfloat16))
        return y.detach().cpu(), xg.grad.cpu(), layer.weight.grad.cpu().reshape(-1), yh.float().cpu()

    y, dx, dw, yh = SimWorld(1).run(body)[0]
    xr = x.clone().requires_grad_(True)
    yr = ref(xr)
    yr.backward(torch.ones_like(yr) * 0.5 + yr.detach())
    assert torch.allclose(y, yr.detach(), rtol=1e-5, atol=1e-5)
    assert torch.allclose(dx, xr.grad, rtol=1e-4, atol=1e-5)
    assert torch.allclose(dw, ref.weight.grad, rtol=1e-4, atol=1e-4)
    assert torch.allclose(yh, yr.detach(), rtol=2e-2, atol=2e-2)


def test_layernorm_large_offset_keeps_accuracy(ops):
    # mean >> std: no fp32 evaluation can hold 1e-5 here (the mean itself is only
    # good to ~1e-4 of a standard deviation); the kernel must be as good as the
    # reference's fp32 sequence, which a one-pass E[x^2]-E[x]^2 would not be
    rng = np.random.default_rng(77)
    shards = [(1000.0 + rng.standard_normal((64, 256))).astype(np.float32) for _ in range(2)]
    _ln_case(ops, shards, None, None, 1e-5, strict=False)


def test_layernorm_layer_matches_torch(golden):
    """DistributedLayerNorm on every worker (loopback) vs torch.nn.LayerNorm on
    the whole tensor: the reference's test, its geometries, its tolerance."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    torch.manual_seed(0)
    # the reference's geometries (all with equal shard widths), then geometries whose normalised dimensions do not
    # divide evenly among the workers, which the reference never tests
    uneven = [{"P_x_shape": [1, 1, 3], "input_shape": [2, 5, 10], "normalized_shape": [10]},
              {"P_x_shape": [2, 1, 2], "input_shape": [5, 3, 7], "normalized_shape": [3, 7]},
              {"P_x_shape": [1, 2, 2], "input_shape": [3, 5, 9], "normalized_shape": [5, 9]},
              {"P_x_shape": [2, 3], "input_shape": [6, 301], "normalized_shape": [301]}]
    seen_uneven = 0
    for geom in golden("layer_geometries.json")["layernorm"] + uneven:
        P, shape, norm = geom["P_x_shape"], geom["input_shape"], geom["normalized_shape"]
        nn_ = len(norm)
        x = torch.rand(shape)
        gamma = 1 + 0.1 * torch.randn(norm)
        beta = 0.1 * torch.randn(norm)
        n = int(np.prod(P))
        xs = o_rep.scatter(x.numpy(), P)
        Pn = [1] * (len(shape) - nn_) + list(P[-nn_:])
        full = [1] * (len(shape) - nn_) + list(norm)
        gs = o_rep.scatter(gamma.numpy().reshape(full), Pn)
        bs = o_rep.scatter(beta.numpy().reshape(full), Pn)

        def body(P_world):
            P_x = P_world.create_partition_inclusive(list(range(n))).create_cartesian_topology_partition(P)
            layer = DistributedLayerNorm(P_x, norm)
            assert (np.asarray(layer.broadcast.P_x.shape) - np.asarray([1] * (len(P) - nn_) + list(P[-nn_:]))).sum() == 0
            red = int(np.ravel_multi_index(tuple(int(i) for i in P_x.index[-nn_:]), tuple(P[-nn_:])))
            with torch.no_grad():
                if layer.P_w.active:
                    layer.weight.copy_(torch.from_numpy(gs[red]))
                    layer.bias.copy_(torch.from_numpy(bs[red]))
                y = layer(torch.from_numpy(xs[P_x.rank]).cuda())
            torch.cuda.synchronize()
            return y.cpu().numpy()

        outs = SimWorld(n).run(body)
        even = not any(s % p for s, p in zip(shape[-nn_:], P[-nn_:]))
        if even:
            want = F.layer_norm(x, tuple(norm), gamma, beta, 1e-5).numpy()
            parts = o_rep.scatter(want, P)
        else:
            # unequal widths: the reference is the mean of local statistics (not the layer norm of the whole
            # row), restated by the oracle over each group of workers that share rows
            seen_uneven += 1
            parts = [None] * n
            lead_shape, red_shape = tuple(P[:len(P) - nn_]), tuple(P[-nn_:])
            n_red = int(np.prod(red_shape))
            for lead in np.ndindex(*lead_shape) if lead_shape else [()]:
                group = [int(np.ravel_multi_index(tuple(lead) + tuple(r), tuple(P))) for r in np.ndindex(*red_shape)]
                res = o_ln.forward_shards([xs[r] for r in group], [gs[k] for k in range(n_red)],
                                          [bs[k] for k in range(n_red)], 1e-5, num_norm_dims=nn_, dtype=np.float64)
                for r, y in zip(group, res):
                    parts[r] = y
        for got, part in zip(outs, parts):
            assert got.shape == part.shape, geom
            assert np.allclose(got, part, rtol=1e-4, atol=1e-5), geom     # reference tolerance is atol sqrt(1e-7)
    assert seen_uneven == len(uneven)


@pytest.mark.parametrize("cols", [[256, 256, 256, 256], [64, 64], [300, 212], [7, 9], [2048], [5000, 40], [4] * 70])
@pytest.mark.parametrize("affine", [True, False])
def test_layernorm_backward_kernels_match_oracle(ops, cols, affine):
    """dx, dgamma, dbeta of one worker of the reduction group; the row sums of
    the other workers come from the oracle.  fp32 kernels against the fp64
    closed form: 1e-5 relative to the gradient's scale."""
    rng = np.random.default_rng(sum(cols) + len(cols))
    rows, eps = 37, 1e-5
    shards = [(rng.standard_normal((rows, c)) * 2 + 0.5).astype(np.float32) for c in cols]
    dys = [rng.standard_normal((rows, c)).astype(np.float32) for c in cols]
    gammas = [(1 + 0.1 * rng.standard_normal(c)).astype(np.float32) if affine else None for c in cols]
    betas = [(0.1 * rng.standard_normal(c)).astype(np.float32) if affine else None for c in cols]
    want_dx, want_dg, want_db = o_ln.backward_shards(shards, gammas, dys, eps)
    P = len(cols)
    for live in {0, P - 1}:
        x2d = torch.from_numpy(shards[live]).cuda()
        dy2d = torch.from_numpy(dys[live]).cuda()
        g = None if not affine else torch.from_numpy(gammas[live]).cuda()
        b = None if not affine else torch.from_numpy(betas[live]).cuda()
        parts = [torch.from_numpy(o_ln.partial_stats(s).astype(np.float32)).cuda() for s in shards]
        parts[live] = ops.ln_partial_stats(x2d)
        _, mean, rstd = ops.ln_normalize_affine(x2d, torch.stack(parts).contiguous(), cols, g, b, eps, want_stats=True)
        sums = ops.ln_backward_partial(dy2d, x2d, mean, rstd, g)
        # the other workers' sums, from the oracle's intermediate quantities (fp64 -> fp32)
        m64 = sum(s.astype(np.float64).mean(axis=1) for s in shards) / P
        v64 = sum(((s.astype(np.float64) - m64[:, None]) ** 2).mean(axis=1) for s in shards) / P
        r64 = 1.0 / np.sqrt(v64 + eps)
        gathered = []
        for p in range(P):
            gp = dys[p].astype(np.float64) * (gammas[p].astype(np.float64) if affine else 1.0)
            xh = (shards[p].astype(np.float64) - m64[:, None]) * r64[:, None]
            pair = np.stack([gp.sum(axis=1), (gp * xh).sum(axis=1)], axis=1)
            if p == live:
                scale = scale_live = np.abs(gp).sum(axis=1).max()
                assert np.allclose(sums.cpu().numpy(), pair, rtol=1e-4, atol=2e-5 * scale)
                gathered.append(sums)
            else:
                gathered.append(torch.from_numpy(pair.astype(np.float32)).cuda())
        dx = ops.ln_backward_input(dy2d, x2d, mean, rstd, g, torch.stack(gathered).contiguous(), 1.0 / (P * cols[live]))
        dg, db = ops.ln_backward_params(dy2d, x2d, mean, rstd)
        torch.cuda.synchronize()
        tol = 1e-5 * max(1.0, np.abs(want_dx[live]).max())
        assert np.abs(dx.cpu().numpy() - want_dx[live]).max() <= 4 * tol
        assert np.allclose(dg.cpu().numpy(), want_dg[live], rtol=1e-4, atol=1e-4)
        assert np.allclose(db.cpu().numpy(), want_db[live], rtol=1e-4, atol=1e-4)
        # the two-launch variant: same sums, same gradients
        sums2, work = ops.ln_backward_partial_params(dy2d, x2d, mean, rstd, g)
        assert np.allclose(sums2.cpu().numpy(), sums.cpu().numpy(), rtol=1e-5, atol=1e-5 * scale_live)
        gathered[live] = sums2
        dx2, dg2, db2 = ops.ln_backward_input_params(dy2d, x2d, mean, rstd, g, torch.stack(gathered).contiguous(),
                                                     1.0 / (P * cols[live]), work)
        torch.cuda.synchronize()
        assert np.abs(dx2.cpu().numpy() - want_dx[live]).max() <= 4 * tol
        assert np.allclose(dg2.cpu().numpy(), want_dg[live], rtol=1e-4, atol=1e-4)
        assert np.allclose(db2.cpu().numpy(), want_db[live], rtol=1e-4, atol=1e-4)
        dx3, dg3, db3 = ops.ln_backward_input_params(dy2d, x2d, mean, rstd, g, torch.stack(gathered).contiguous(),
                                                     1.0 / (P * cols[live]), work, want_gamma=False, want_beta=True)
        assert dg3 is None and torch.equal(db3, db2) and torch.equal(dx3, dx2)
        # one pass over dy and x, the other workers' sums in memory beforehand: the same results, own sums written in place
        table = torch.stack(gathered).contiguous()
        if ops.ln_backward_one_pass_supported(dy2d, x2d, g, P):
            poisoned = table.clone()
            poisoned[live] = float("nan")
            dx4, dg4, db4 = ops.ln_backward_one_pass(dy2d, x2d, mean, rstd, g, 1.0 / (P * cols[live]), poisoned, live)
            torch.cuda.synchronize()
            assert torch.equal(poisoned, table)
            assert torch.equal(dx4, dx2) and torch.equal(dg4, dg2) and torch.equal(db4, db2)
        else:
            with pytest.raises(RuntimeError, match="code -5"):
                ops.ln_backward_one_pass(dy2d, x2d, mean, rstd, g, 1.0 / (P * cols[live]), table.clone(), live)


@pytest.mark.parametrize("rows,cols", [(1, 4), (37, 256), (300, 1024), (1000, 300), (5000, 64), (33, 1028)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_norm_backward_of_whole_rows_in_one_pass(ops, rows, cols, dtype):
    """Rows one worker holds whole (the backward of the reference's
    F.layer_norm branch, nn/layernorm.py:319): dx, dgamma, dbeta from one pass
    over dy and x against torch autograd in float64, and against the two
    launches bit for bit."""
    gen = torch.Generator().manual_seed(rows * 7 + cols)
    x = (torch.randn(rows, cols, generator=gen) * 2 + 0.3).to(dtype)
    dy = torch.randn(rows, cols, generator=gen).to(dtype)
    gamma = (1 + 0.1 * torch.randn(cols, generator=gen)).to(dtype)
    beta = (0.1 * torch.randn(cols, generator=gen)).to(dtype)
    xg, dyg, gg, bg = x.cuda(), dy.cuda(), gamma.cuda(), beta.cuda()
    _, mean, rstd = ops.layer_norm(xg, gg, bg, 1e-5, want_stats=True)
    if not ops.ln_backward_one_pass_supported(dyg, xg, gg):
        assert cols > 1024
        with pytest.raises(RuntimeError, match="code -5"):
            ops.ln_backward_one_pass(dyg, xg, mean, rstd, gg, 1.0 / cols)
        return
    dx, dg, db = ops.ln_backward_one_pass(dyg, xg, mean, rstd, gg, 1.0 / cols)
    sums, work = ops.ln_backward_partial_params(dyg, xg, mean, rstd, gg)
    dx2, dg2, db2 = ops.ln_backward_input_params(dyg, xg, mean, rstd, gg, sums.unsqueeze(0).contiguous(), 1.0 / cols, work)
    torch.cuda.synchronize()
    assert torch.equal(dx.view(torch.uint8), dx2.view(torch.uint8))
    assert torch.equal(dg.view(torch.uint8), dg2.view(torch.uint8)) and torch.equal(db.view(torch.uint8), db2.view(torch.uint8))
    xr = x.double().requires_grad_(True)
    gr, br = gamma.double().requires_grad_(True), beta.double().requires_grad_(True)
    F.layer_norm(xr, (cols,), gr, br, 1e-5).backward(dy.double())
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7
    scale = max(1.0, float(xr.grad.abs().max()))
    assert float((dx.cpu().double() - xr.grad).abs().max()) <= 4 * tol * scale
    assert torch.allclose(dg.cpu().double(), gr.grad, rtol=10 * tol, atol=10 * tol * max(1.0, float(gr.grad.abs().max())))
    assert torch.allclose(db.cpu().double(), br.grad, rtol=10 * tol, atol=10 * tol * max(1.0, float(br.grad.abs().max())))
    # without parameter gradients: dx alone, no second launch
    dx5, dg5, db5 = ops.ln_backward_one_pass(dyg, xg, mean, rstd, gg, 1.0 / cols, want_gamma=False, want_beta=False)
    assert dg5 is None and db5 is None and torch.equal(dx5, dx)


@pytest.mark.parametrize("cols", [1, 2, 3, 5, 255, 257, 511, 514, 1023, 1027, 2047, 2049, 4095, 4098, 8191, 8193, 16383, 16385])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_layer_norm_rows_of_any_length_and_address(ops, dtype, cols):
    """Rows that are no multiple of four elements, whole and split over two workers, at the widths where the kernel's shape
    changes: rows with an odd pitch that start one element into their buffer and end where it ends, whose neighbours hold
    NaN, against float64; what lies between the rows of the output stays untouched."""
    rows, pad = 7, 3
    gen = torch.Generator().manual_seed(cols)
    x = (torch.randn(rows, cols, generator=gen) * 2 + 0.5).to(dtype)
    gamma = (1 + 0.1 * torch.randn(cols, generator=gen)).to(dtype)
    beta = (0.1 * torch.randn(cols, generator=gen)).to(dtype)
    store = torch.full((1 + rows * (cols + pad) - pad,), float("nan"), dtype=dtype, device="cuda")
    xg = store[1:].as_strided((rows, cols), (cols + pad, 1), 1)
    xg.copy_(x)
    shifted = [torch.empty(cols + 1, dtype=dtype, device="cuda")[1:].copy_(t) for t in (gamma, beta)]
    y, mean, rstd = ops.layer_norm(xg, *shifted, 1e-3, want_stats=True)
    stats = ops.ln_partial_stats(xg)
    other = torch.stack([torch.full((rows,), 0.25), torch.full((rows,), 3.0)], dim=1).cuda()
    y2 = ops.ln_normalize_affine(xg, torch.stack([stats, other]).contiguous(), [cols, 5], *shifted, 1e-3)
    x64 = x.double()
    m, q = x64.mean(1), ((x64 - x64.mean(1, keepdim=True)) ** 2).sum(1)
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]

    def check(got, want, size):     # one rounding of the result and a few units of fp32 sums
        assert bool(((got.cpu().double() - want).abs() <= ulp * want.abs() + 4e-6 * size).all())
    assert bool(((stats.cpu().double()[:, 0] - m).abs() <= 4e-6 * 4).all()) and bool(((stats.cpu().double()[:, 1] - q).abs() <= 4e-6 * (q + 4)).all())
    check(y, (x64 - m[:, None]) / (q / cols + 1e-3).sqrt()[:, None] * gamma.double() + beta.double(), 8.0 * (1 + float((q / cols + 1e-3).rsqrt().max())))
    m2 = (m + 0.25) / 2
    v2 = (q / cols + (m - m2) ** 2 + 3.0 / 5 + (0.25 - m2) ** 2) / 2
    check(y2, (x64 - m2[:, None]) / (v2 + 1e-3).sqrt()[:, None] * gamma.double() + beta.double(), 8.0)


@pytest.mark.parametrize("rows,cols,pad", [(1, 2052, 0), (3, 2056, 4), (4097, 2052, 4), (8191, 2056, 0), (9001, 4096, 0), (70, 4100, 0),
                                           (5000, 8192, 8), (33, 8196, 0), (2100, 8200, 0), (1025, 16384, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_layer_norm_of_long_rows_walked_by_workgroups(ops, dtype, rows, cols, pad):
    """Rows a workgroup holds in pieces of four and eight elements, where a workgroup has one row, several, and one less than
    the others: y, mean and rstd against float64, with a pitch and a row of infinities that must not reach its neighbours;
    the statistics alone, and statistics and result in one launch, give the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = (torch.randn(rows, cols + pad, generator=gen, device="cuda") * 2 + 0.5).to(dtype)[:, :cols]
    gamma = (1 + 0.1 * torch.randn(cols, generator=gen, device="cuda")).to(dtype)
    beta = (0.1 * torch.randn(cols, generator=gen, device="cuda")).to(dtype)
    bad = rows // 2
    if rows > 1:
        x[bad, 1] = float("inf")
    y, mean, rstd = ops.layer_norm(x, gamma, beta, 1e-3, want_stats=True)
    stats = ops.ln_partial_stats(x)
    pairs = torch.stack([torch.zeros_like(stats), stats]).contiguous()
    joined = pairs.clone()
    joined[1] = 0
    two = ops.ln_normalize_affine(x, pairs, [cols, cols], gamma, beta, 1e-3)
    one = ops.ln_stats_normalize(x, joined, 1, [cols, cols], gamma, beta, 1e-3)
    keep = torch.ones(rows, dtype=torch.bool, device="cuda")
    if rows > 1:
        keep[bad] = False
        assert bool(y[bad].isnan().any()) and not bool(y[keep].isnan().any())
    assert torch.equal(joined[1][keep], stats[keep]) and torch.equal(one[keep], two[keep])
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for part in keep.nonzero().flatten().split(1024):
        x64 = x[part].double()
        m = x64.mean(1)
        r = ((x64 - m[:, None]).square().mean(1) + 1e-3).rsqrt()
        want = (x64 - m[:, None]) * r[:, None] * gamma.double() + beta.double()
        # one rounding of the result and a few units of fp32 sums (values up to 12, |x| rstd up to 6)
        assert bool(((y[part].double() - want).abs() <= ulp * want.abs() + 4e-6 * 8).all())
        assert bool(((mean[part].double() - m).abs() <= 4e-6 * 4).all()) and bool(((rstd[part].double() - r).abs() <= 4e-6 * r).all())


@pytest.mark.parametrize("rows,cols", [(3, 256), (1, 257), (70, 511), (33, 512), (65, 516), (9, 1023), (40, 1024), (5, 1025), (1, 2049),
                                       (9, 2050), (70, 2055), (1030, 4093), (300, 8185), (5, 8193), (6, 16383)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shift,pad", [(0, 0), (1, 0), (3, 5)])
def test_layer_norm_of_long_rows_at_any_address(ops, dtype, rows, cols, shift, pad):
    """Rows that end inside a piece, at any address and pitch: y, the statistics, the backward's row sums and dx against
    float64; nothing next to the rows is written, and infinities stay in their row."""
    gen = torch.Generator(device="cuda").manual_seed(rows + cols)

    def at(rows, cols, pad, scale, offset):
        pool = (torch.randn(rows * (cols + pad) + shift + 8, generator=gen, device="cuda") * scale + offset).to(dtype)
        return pool[shift:shift + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]

    x, dy = at(rows, cols, pad, 2, 0.5), at(rows, cols, pad, 1, 0)
    gamma, beta = at(1, cols, 0, 0.1, 1)[0], at(1, cols, 0, 0.1, 0)[0]
    bad = rows - 1
    keep = torch.ones(rows, dtype=torch.bool, device="cuda")
    if rows > 1:
        x[bad, cols - 1] = float("inf")
        keep[bad] = False
    y, mean, rstd = ops.layer_norm(x, gamma, beta, 1e-3, want_stats=True)
    stats = ops.ln_partial_stats(x)
    two = ops.ln_normalize_affine(x, torch.stack([stats, stats]), [cols, cols], gamma, beta, 1e-3)
    sums = ops.ln_backward_partial(dy, x, mean, rstd, gamma)
    dx = ops.ln_backward_input(dy, x, mean, rstd, gamma, torch.stack([sums, sums]), 0.5 / cols)
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for part in keep.nonzero().flatten().split(512):
        x64, d64 = x[part].double(), dy[part].double()
        m = x64.mean(1, keepdim=True)
        r = ((x64 - m).square().mean(1, keepdim=True) + 1e-3).rsqrt()
        h = (x64 - m) * r
        want = h * gamma.double() + beta.double()
        # one rounding of the result and a few units of fp32 sums (values up to 12, |x| rstd up to 6)
        assert bool(((y[part].double() - want).abs() <= ulp * want.abs() + 4e-6 * 8).all())
        assert bool(((two[part].double() - want).abs() <= ulp * want.abs() + 4e-6 * 8).all())
        assert bool(((mean[part].double() - m[:, 0]).abs() <= 4e-6 * 4).all()) and bool(((rstd[part].double() - r[:, 0]).abs() <= 4e-6 * r[:, 0]).all())
        g = d64 * gamma.double()
        s1, s2 = g.sum(1, keepdim=True), (g * h).sum(1, keepdim=True)
        # fp32 sums of cols terms in 64 lanes of fours: a chain of cols / 256 additions and ten more, of |g| and |g h|
        unit = 2.0 ** -24 * (cols / 256 + 10)
        assert bool(((sums[part, :1].double() - s1).abs() <= unit * g.abs().sum(1, keepdim=True)).all())
        assert bool(((sums[part, 1:].double() - s2).abs() <= (unit + 8e-6) * (g.abs() * (h.abs() + 1)).sum(1, keepdim=True)).all())
        want = r * (g - (s1 + h * s2) / cols)
        assert bool(((dx[part].double() - want).abs() <= ulp * want.abs() + 4e-6 * (g.abs() * r + 1)).all())
    if rows > 1:
        assert bool(y[bad].isnan().any()) and bool(dx[bad].isnan().any())
        assert not bool(y[keep].isnan().any()) and not bool(dx[keep].isnan().any())


@pytest.mark.parametrize("rows,cols,pad", [(1, 1028, 0), (5, 1025, 0), (37, 2048, 4), (3, 2052, 0), (66, 4096, 1), (1029, 4097, 0),
                                           (9, 8192, 0), (7, 8191, 0), (6, 8196, 0), (10, 16384, 8), (8200, 1032, 0),
                                           (1, 513, 0), (70, 514, 3), (65, 1023, 0), (300, 768, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_layer_norm_backward_of_long_whole_rows(ops, rows, cols, pad, dtype):
    """Rows a workgroup owns: dx, dgamma and dbeta in one pass against float64 autograd of the same inputs, at the widths
    where the kernel's shape changes, aligned and not, with a pitch, with one row per split and with several; and the row
    sums and column sums of the split form (a split per CU from 8161 rows on)."""
    gen = torch.Generator().manual_seed(rows * 7 + cols)
    store = torch.randn(2, rows, cols + pad, generator=gen).to(dtype)
    x, dy = store[0, :, :cols], store[1, :, :cols]
    gamma = (1 + 0.1 * torch.randn(cols, generator=gen)).to(dtype)
    beta = torch.zeros(cols).to(dtype)
    sg, gg = store.cuda(), gamma.cuda()
    xg, dyg = sg[0, :, :cols], sg[1, :, :cols]
    _, mean, rstd = ops.layer_norm(xg, gg, beta.cuda(), 1e-5, want_stats=True)
    assert ops.ln_backward_whole_rows_supported(dyg, xg, gg)
    dx, dg, db = ops.ln_backward_whole_rows(dyg, xg, mean, rstd, gg, 1.0 / cols)
    only_dx = ops.ln_backward_whole_rows(dyg, xg, mean, rstd, gg, 1.0 / cols, want_gamma=False, want_beta=False)
    assert torch.equal(only_dx[0], dx) and only_dx[1] is None and only_dx[2] is None
    sums, work = ops.ln_backward_partial_params(dyg, xg, mean, rstd, gg)
    dx2, dg2, db2 = ops.ln_backward_input_params(dyg, xg, mean, rstd, gg, sums.unsqueeze(0).contiguous(), 1.0 / cols, work)
    xr, gr, br = x.double().requires_grad_(True), gamma.double().requires_grad_(True), beta.double().requires_grad_(True)
    F.layer_norm(xr, (cols,), gr, br, 1e-5).backward(dy.double())
    # one rounding of the result (half a unit in the last of 24, 8 or 11 bits: 2^-24, 2^-8, 2^-11 of it), and fp32 sums: a
    # few units of the sums' size (dx: of its terms; parameters: sqrt(rows) of dy xhat)
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got_dx, got_dg, got_db in ((dx, dg, db), (dx2, dg2, db2)):
        for got, want, size in ((got_dx, xr.grad, 4.0), (got_dg, gr.grad, 4.0 * rows ** 0.5), (got_db, br.grad, 4.0 * rows ** 0.5)):
            err = (got.cpu().double() - want).abs()
            assert bool((err <= ulp * want.abs() + 2e-6 * size).all()), float(err.max())


@pytest.mark.parametrize("rows,cols,pad", [(1, 1025, 0), (4, 8192, 0), (5, 1028, 3), (509, 1026, 0), (513, 2049, 1), (1023, 1536, 0), (1025, 1100, 0),
                                           (2049, 1025, 0), (9, 8193, 0), (3, 1024, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_norm_row_and_column_sums_in_one_pass(ops, rows, cols, pad, dtype):
    """Row sums and column sums of shared rows where the number of row splits changes, with the room that the layer hands
    over and with room for fewer splits and for one, against float64."""
    gen = torch.Generator().manual_seed(rows * 11 + cols)
    store = torch.randn(2, rows, cols + pad, generator=gen).to(dtype)
    gamma = (1 + 0.1 * torch.randn(cols, generator=gen)).to(dtype)
    mean, rstd = 0.1 * torch.randn(rows, generator=gen), 1 + 0.1 * torch.rand(rows, generator=gen)
    x, dy = store[0, :, :cols].double(), store[1, :, :cols].double()
    xhat = (x - mean.double()[:, None]) * rstd.double()[:, None]
    g = dy * gamma.double()
    want = ((g.sum(1), 4 * cols ** 0.5), ((g * xhat).sum(1), 4 * cols ** 0.5), ((dy * xhat).sum(0), 4 * rows ** 0.5), (dy.sum(0), 4 * rows ** 0.5))
    sg, gg, mg, rg = store.cuda(), gamma.cuda(), mean.cuda(), rstd.cuda()
    xg, dyg = sg[0, :, :cols], sg[1, :, :cols]
    from distdl_amd import _lib
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    code = _lib.DDL_DT_F32 if dtype == torch.float32 else _lib.DDL_DT_BF16
    ulp = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -8
    def by_hand(room):   # ddl_* with room for as many splits
        sums, work = torch.empty(rows, 2, device="cuda"), torch.empty(2 * room * cols, device="cuda")
        dx, dg, db = torch.empty(rows, cols, dtype=dtype, device="cuda"), torch.empty_like(gg), torch.empty_like(gg)
        at = (dyg.data_ptr(), xg.data_ptr(), code, rows, cols, cols + pad, cols + pad, mg.data_ptr(), rg.data_ptr(), gg.data_ptr())
        assert lib.ddl_ln_bwd_partial_params(*at, sums.data_ptr(), work.data_ptr(), work.numel(), stream) == 0
        assert lib.ddl_ln_bwd_input_params(*at, sums.data_ptr(), 1, 1.0 / cols, dx.data_ptr(), cols, work.data_ptr(), work.numel(), dg.data_ptr(),
                                           db.data_ptr(), stream) == 0
        return sums, dg, db
    def by_layer():
        sums, work = ops.ln_backward_partial_params(dyg, xg, mg, rg, gg)
        return (sums, *ops.ln_backward_input_params(dyg, xg, mg, rg, gg, sums.unsqueeze(0).contiguous(), 1.0 / cols, work)[1:])
    for sums, dg, db in (by_layer(), by_hand(256), by_hand((rows + 31) // 32), by_hand(1)):
        # fp32 sums of terms around one: a few units of sqrt(terms); parameters rounded once to their type
        for (value, size), got, rounding in zip(want, (sums[:, 0], sums[:, 1], dg, db), (0, 0, ulp, ulp)):
            err = (got.cpu().double() - value).abs()
            assert bool((err <= rounding * value.abs() + 2e-6 * size).all()), float(err.max())


@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("cols", [[256, 256], [300, 212], [7, 9], [2048], [1030]])
def test_layernorm_backward_16_bit_elements(ops, dtype, ulp, cols):
    """The backward kernels on bf16 / fp16 tensors: arithmetic in fp32 on the
    16-bit values, one rounding when dx, dgamma and dbeta are stored -- so the
    results must be the fp64 closed form of the same 16-bit inputs to within one
    rounding of the result type (plus fp32 summation noise)."""
    rng = np.random.default_rng(sum(cols) + 5)
    rows, eps = 45, 1e-5
    def q(a):   # through the 16-bit type and back
        return torch.from_numpy(a.astype(np.float32)).to(dtype)
    shards = [q(rng.standard_normal((rows, c)) * 2 + 0.5) for c in cols]
    dys = [q(rng.standard_normal((rows, c))) for c in cols]
    gammas = [q(1 + 0.1 * rng.standard_normal(c)) for c in cols]
    f64 = lambda t: t.double().numpy()
    want_dx, want_dg, want_db = o_ln.backward_shards([f64(t) for t in shards], [f64(t) for t in gammas], [f64(t) for t in dys], eps)
    P = len(cols)
    m64 = sum(f64(s).mean(axis=1) for s in shards) / P
    v64 = sum(((f64(s) - m64[:, None]) ** 2).mean(axis=1) for s in shards) / P
    r64 = 1.0 / np.sqrt(v64 + eps)
    live = P - 1
    x2d, dy2d, g = shards[live].cuda(), dys[live].cuda(), gammas[live].cuda()
    parts = [torch.from_numpy(o_ln.partial_stats(f64(s)).astype(np.float32)).cuda() for s in shards]
    parts[live] = ops.ln_partial_stats(x2d)
    _, mean, rstd = ops.ln_normalize_affine(x2d, torch.stack(parts).contiguous(), cols, g, g, eps, want_stats=True)
    assert mean.dtype == torch.float32 and rstd.dtype == torch.float32
    gathered = []
    for p in range(P):
        gp = f64(dys[p]) * f64(gammas[p])
        xh = (f64(shards[p]) - m64[:, None]) * r64[:, None]
        gathered.append(torch.from_numpy(np.stack([gp.sum(axis=1), (gp * xh).sum(axis=1)], axis=1).astype(np.float32)).cuda())
    sums = ops.ln_backward_partial(dy2d, x2d, mean, rstd, g)
    scale = np.abs(f64(dys[live]) * f64(gammas[live])).sum(axis=1).max()
    assert np.allclose(sums.cpu().numpy(), gathered[live].cpu().numpy(), rtol=1e-4, atol=2e-5 * scale)
    gathered[live] = sums
    stack = torch.stack(gathered).contiguous()
    weight = 1.0 / (P * cols[live])
    dx = ops.ln_backward_input(dy2d, x2d, mean, rstd, g, stack, weight)
    dg, db = ops.ln_backward_params(dy2d, x2d, mean, rstd)
    sums2, work = ops.ln_backward_partial_params(dy2d, x2d, mean, rstd, g)
    gathered[live] = sums2
    dx2, dg2, db2 = ops.ln_backward_input_params(dy2d, x2d, mean, rstd, g, torch.stack(gathered).contiguous(), weight, work)
    torch.cuda.synchronize()
    for got_dx, got_dg, got_db in ((dx, dg, db), (dx2, dg2, db2)):
        assert got_dx.dtype == dtype and got_dg.dtype == dtype and got_db.dtype == dtype
        for got, want in ((got_dx, want_dx[live]), (got_dg, want_dg[live]), (got_db, want_db[live])):
            err = np.abs(got.double().cpu().numpy() - want)
            assert (err <= ulp * np.abs(want) + 1e-4 * max(1.0, np.abs(want).max())).all(), float(err.max())
    # misaligned rows (odd pitch) take the element-wise kernels: same values
    pitch = cols[live] + 3
    xp = torch.zeros((rows, pitch), dtype=dtype, device="cuda")
    dyp = torch.zeros((rows, pitch), dtype=dtype, device="cuda")
    xp[:, :cols[live]] = x2d
    dyp[:, :cols[live]] = dy2d
    dx3 = ops.ln_backward_input(dyp[:, :cols[live]], xp[:, :cols[live]], mean, rstd, g, stack, weight)
    err = np.abs(dx3.double().cpu().numpy() - want_dx[live])
    assert (err <= ulp * np.abs(want_dx[live]) + 1e-4 * max(1.0, np.abs(want_dx[live]).max())).all()


def test_layernorm_layer_backward_in_bfloat16():
    """The layer in bfloat16 on two workers that share the rows, forward and
    backward through autograd, against torch's layer norm in float64 on the
    same bfloat16 values."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    torch.manual_seed(11)
    P, shape, norm = [1, 1, 2], [4, 6, 128], [128]
    x = torch.randn(shape).to(torch.bfloat16)
    dy = torch.randn(shape).to(torch.bfloat16)
    gamma = (1 + 0.1 * torch.randn(norm)).to(torch.bfloat16)
    beta = (0.1 * torch.randn(norm)).to(torch.bfloat16)

    def body(P_world):
        P_x = P_world.create_partition_inclusive([0, 1]).create_cartesian_topology_partition(P)
        layer = DistributedLayerNorm(P_x, norm, dtype=torch.bfloat16)
        half = slice(64 * P_x.rank, 64 * P_x.rank + 64)
        with torch.no_grad():
            layer.weight.copy_(gamma[half].reshape(1, 1, 64))
            layer.bias.copy_(beta[half].reshape(1, 1, 64))
        xin = x[..., half].contiguous().cuda().requires_grad_(True)
        y = layer(xin)
        y.backward(dy[..., half].contiguous().cuda())
        torch.cuda.synchronize()
        assert y.dtype == torch.bfloat16 and xin.grad.dtype == torch.bfloat16 and layer.weight.grad.dtype == torch.bfloat16
        return y.detach().cpu(), xin.grad.cpu(), layer.weight.grad.cpu().reshape(-1), layer.bias.grad.cpu().reshape(-1)

    outs = SimWorld(2).run(body)
    xr, gr, br = x.double().requires_grad_(True), gamma.double().requires_grad_(True), beta.double().requires_grad_(True)
    yr = F.layer_norm(xr, tuple(norm), gr, br, 1e-5)
    yr.backward(dy.double())
    for rank, (y, dx, dw, db) in enumerate(outs):
        half = slice(64 * rank, 64 * rank + 64)
        for got, want in ((y, yr.detach()[..., half]), (dx, xr.grad[..., half]), (dw, gr.grad[half]), (db, br.grad[half])):
            err = (got.double() - want).abs()
            assert (err <= 2.0 ** -8 * want.abs() + 1e-3 * max(1.0, float(want.abs().max()))).all(), float(err.max())


def test_layernorm_backward_two_launch_variant_many_rows(ops):
    """Row splits of more than one wavefront round, a last split that is short,
    rows of 256 / 512 / 1024 floats (one, two, four vectors per lane)."""
    rng = np.random.default_rng(77)
    for rows, cols in ((8192, 256), (1000, 512), (333, 1024), (70, 1028)):
        x = (rng.standard_normal((rows, cols)) * 1.5 + 0.25).astype(np.float32)
        dy = rng.standard_normal((rows, cols)).astype(np.float32)
        gamma = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
        want_dx, want_dg, want_db = o_ln.backward_shards([x], [gamma], [dy], 1e-5)
        xg, dyg, gg = torch.from_numpy(x).cuda(), torch.from_numpy(dy).cuda(), torch.from_numpy(gamma).cuda()
        stats = ops.ln_partial_stats(xg)
        _, mean, rstd = ops.ln_normalize_affine(xg, stats.unsqueeze(0).contiguous(), [cols], gg, gg, 1e-5, want_stats=True)
        sums, work = ops.ln_backward_partial_params(dyg, xg, mean, rstd, gg)
        dx, dg, db = ops.ln_backward_input_params(dyg, xg, mean, rstd, gg, sums.unsqueeze(0).contiguous(), 1.0 / cols, work)
        torch.cuda.synchronize()
        tol = 1e-5 * max(1.0, np.abs(want_dx[0]).max())
        assert np.abs(dx.cpu().numpy() - want_dx[0]).max() <= 4 * tol
        scale = np.sqrt(rows)
        assert np.allclose(dg.cpu().numpy(), want_dg[0], rtol=1e-4, atol=1e-4 * scale)
        assert np.allclose(db.cpu().numpy(), want_db[0], rtol=1e-4, atol=1e-4 * scale)


def test_layernorm_layer_backward_matches_torch():
    """DistributedLayerNorm on every worker (loopback), forward and backward,
    against torch.nn.functional.layer_norm on the whole tensor."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    torch.manual_seed(5)
    P, shape, norm = [1, 2, 2], [3, 8, 64], [64]
    x = torch.randn(shape)
    dy = torch.randn(shape)
    gamma = 1 + 0.1 * torch.randn(norm)
    beta = 0.1 * torch.randn(norm)
    xs, dys = o_rep.scatter(x.numpy(), P), o_rep.scatter(dy.numpy(), P)
    gs = o_rep.scatter(gamma.numpy().reshape(1, 1, 64), [1, 1, 2])
    bs = o_rep.scatter(beta.numpy().reshape(1, 1, 64), [1, 1, 2])

    def body(P_world):
        P_x = P_world.create_partition_inclusive(list(range(4))).create_cartesian_topology_partition(P)
        layer = DistributedLayerNorm(P_x, norm)
        red = int(P_x.index[-1])
        with torch.no_grad():
            if layer.P_w.active:
                layer.weight.copy_(torch.from_numpy(gs[red]))
                layer.bias.copy_(torch.from_numpy(bs[red]))
        xin = torch.from_numpy(xs[P_x.rank]).cuda().requires_grad_(True)
        y = layer(xin)
        y.backward(torch.from_numpy(dys[P_x.rank]).cuda())
        torch.cuda.synchronize()
        wgrad = layer.weight.grad.cpu().numpy() if layer.P_w.active and layer.weight.grad is not None else None
        bgrad = layer.bias.grad.cpu().numpy() if layer.P_w.active and layer.bias.grad is not None else None
        return xin.grad.cpu().numpy(), wgrad, bgrad, tuple(int(i) for i in P_x.index)

    outs = SimWorld(4).run(body)
    xr, gr, br = x.clone().requires_grad_(True), gamma.clone().requires_grad_(True), beta.clone().requires_grad_(True)
    F.layer_norm(xr, tuple(norm), gr, br, 1e-5).backward(dy)
    want_dx = o_rep.scatter(xr.grad.numpy(), P)
    for rank, (dx, wgrad, bgrad, index) in enumerate(outs):
        assert np.allclose(dx, want_dx[rank], rtol=1e-4, atol=1e-5)
    # parameter gradients: summed over the workers that share a feature shard
    for red in range(2):
        lo, hi = 32 * red, 32 * (red + 1)
        got_w = [o[1] for o in outs if o[1] is not None and o[3][-1] == red]
        got_b = [o[2] for o in outs if o[2] is not None and o[3][-1] == red]
        assert got_w and got_b
        assert np.allclose(sum(g.reshape(-1) for g in got_w), gr.grad.numpy()[lo:hi], rtol=1e-4, atol=1e-4)
        assert np.allclose(sum(g.reshape(-1) for g in got_b), br.grad.numpy()[lo:hi], rtol=1e-4, atol=1e-4)


def test_layernorm_training_step_reference_cases(golden):
    """The reference's test_batch_norm_with_training (tests/layers/test_layernorm.py:143-277)
    on its ten geometries: scatter from one worker, DistributedLayerNorm, gather,
    squared-error loss, backward, a parameter step, a second forward -- against
    torch.nn.LayerNorm on the whole tensor with the reference's tolerances
    (rtol 1e-4, atol sqrt(1e-7)); the parameter gradients, which the reference
    collects but never compares, are compared here as well."""
    import math

    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm, Repartition
    from distdl_amd.utilities.torch import zero_volume_tensor
    rtol, atol = 1e-4, math.sqrt(1e-7)
    for geom in golden("layer_geometries.json")["layernorm"]:
        P, shape, norm = geom["P_x_shape"], geom["input_shape"], geom["normalized_shape"]
        n, nn_ = int(np.prod(P)), len(norm)
        torch.manual_seed(0)
        x_train, x_eval, target = torch.rand(shape), torch.rand(shape), torch.rand(shape)
        seq = torch.nn.LayerNorm(norm)
        seq_out1 = seq(x_train)
        seq_loss = ((seq_out1 - target) ** 2).sum()
        seq_loss.backward()
        seq_grads = [p.grad.detach().clone() for p in seq.parameters()]
        with torch.no_grad():
            for p in seq.parameters():
                p.copy_(p + 0.1 * p.grad)
            seq_out2 = seq(x_eval)
        Pn = [1] * (len(shape) - nn_) + list(P[-nn_:])
        full = [1] * (len(shape) - nn_) + list(norm)
        want_grads = [o_rep.scatter(g.numpy().reshape(full), Pn) for g in seq_grads]

        def body(P_world):
            P_root = P_world.create_partition_inclusive([0]).create_cartesian_topology_partition([1] * len(shape))
            P_x = P_world.create_partition_inclusive(list(range(n))).create_cartesian_topology_partition(P)
            scatter, gather = Repartition(P_root, P_x), Repartition(P_x, P_root)
            layer = DistributedLayerNorm(P_x, norm)

            def held(t):
                return t.cuda() if P_root.active else zero_volume_tensor(device="cuda")
            layer.train()
            out1 = gather(layer(scatter(held(x_train))))
            loss = ((out1 - held(target)) ** 2).sum()
            assert loss.requires_grad
            loss.backward()
            grads = None
            if layer.P_w.active:
                grads = [p.grad.detach().cpu().numpy().copy() for p in layer.parameters()]
                with torch.no_grad():
                    for p in layer.parameters():
                        p.copy_(p + 0.1 * p.grad)
            layer.eval()
            out2 = gather(layer(scatter(held(x_eval)))).detach()
            torch.cuda.synchronize()
            red = int(np.ravel_multi_index(tuple(int(i) for i in P_x.index[-nn_:]), tuple(P[-nn_:])))
            return out1.detach().cpu(), loss.detach().cpu(), grads, red, out2.cpu()

        outs = SimWorld(n).run(body)
        out1, loss, _, _, out2 = outs[0]
        assert out1.shape == seq_out1.shape and torch.allclose(out1, seq_out1.detach(), rtol=rtol, atol=atol), geom
        assert torch.allclose(loss, seq_loss.detach(), rtol=rtol, atol=atol), geom
        assert out2.shape == seq_out2.shape and torch.allclose(out2, seq_out2, rtol=rtol, atol=atol), geom
        holders = 0
        for _, _, grads, red, _ in outs:
            if grads is None:
                continue
            holders += 1
            assert len(grads) == 2
            for got, want in zip(grads, want_grads):
                assert got.shape == want[red].shape and np.allclose(got, want[red], rtol=rtol, atol=atol), geom
        assert holders == int(np.prod(P[-nn_:])), geom


# ---------------------------------------------------------------- Embedding --

def test_embedding_config3_rank0_bit_exact(ops):
    """Table 128256 x 4096 bf16 split 8-way by vocabulary: rank 0 holds rows
    [0,16032); ids [32,4096] int64 uniform over the whole vocabulary."""
    gen = torch.Generator().manual_seed(1003)
    table = (0.02 * torch.randn(16032, 4096, generator=gen)).to(torch.bfloat16)
    ids = torch.randint(0, 128256, (32, 4096), generator=gen)
    out = ops.embedding_gather(table.cuda(), ids.cuda(), 0, 16032)
    torch.cuda.synchronize()
    assert out.shape == (32, 4096, 4096) and out.dtype == torch.bfloat16
    tb = bits16(table)
    # oracle on a slice of the batch (the whole output is 1 GiB) ...
    got = bits16(out[:2])
    assert np.array_equal(got, o_emb.gather(tb, ids[:2].numpy(), 0, 16032))
    # ... and size-independent properties on all of it
    hit = (ids < 16032)
    assert 0 < int(hit.sum()) < ids.numel()
    out_i = out.view(torch.int16)
    assert int((out_i[~hit.cuda()] != 0).sum()) == 0                       # misses are zero rows
    ref = F.embedding(ids.clamp(max=16031).cuda(), table.cuda()).view(torch.int16)
    assert torch.equal(out_i[hit.cuda()], ref[hit.cuda()])                 # hits are the table rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float64, torch.uint8])
@pytest.mark.parametrize("dim", [1, 3, 8, 100, 512, 1000, 4100])
@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_embedding_small_cases(ops, dtype, dim, idt):
    gen = torch.Generator().manual_seed(dim)
    es = torch.empty((), dtype=dtype).element_size()
    table = torch.randint(0, 256, (23, dim, es), dtype=torch.uint8, generator=gen).view(dtype).reshape(23, dim)
    ids = torch.randint(0, 40, (5, 9), generator=gen).to(idt)
    lo, hi = 7, 30
    out = ops.embedding_gather(table.cuda(), ids.cuda(), lo, hi)
    np_view = {1: np.uint8, 2: np.uint16, 4: np.uint32, 8: np.uint64}[es]
    tb = table.contiguous().view(torch.uint8).numpy().view(np_view).reshape(23, dim)
    got = out.cpu().contiguous().view(torch.uint8).numpy().view(np_view).reshape(5, 9, dim)
    assert np.array_equal(got, o_emb.gather(tb, ids.numpy(), lo, hi))


def test_embedding_layer_full_window_matches_torch():
    """The reference's layer: table split along the embedding dimension, every
    id hits; compared with torch.nn.functional.embedding (tests/layers/test_embedding.py:81-156)."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedEmbedding
    torch.manual_seed(4)
    table = torch.randn(50, 24)
    ids = torch.randint(0, 50, (3, 11))
    want = F.embedding(ids, table)

    def body(P_world):
        P_x = P_world.create_partition_inclusive([0, 1, 2, 3]).create_cartesian_topology_partition([1, 1, 4])
        layer = DistributedEmbedding(P_x, 50, 24)
        assert tuple(layer.P_weight.shape) == (1, 1, 4)
        with torch.no_grad():
            layer.weight.copy_(table[:, 6 * P_x.rank:6 * (P_x.rank + 1)])
            return layer(ids.cuda()).cpu()

    outs = SimWorld(4).run(body)
    assert torch.equal(torch.cat(outs, dim=-1), want)


def test_embedding_backward_as_many_long_rows_in_a_segment_as_there_can_be(ops):
    """255 rows of 513 tokens each, 256 rows apart, so that one workgroup of the bucketing has all of them in its segment and
    orders every bucket by a bit per token number; sums in the order of the tokens, so repeated calls agree bit for bit."""
    rows, dim, tokens = 5 + 256 * 254 + 40, 20, 131072
    gen = torch.Generator(device="cuda").manual_seed(11)
    ids = (5 + 256 * (torch.arange(tokens, device="cuda") % 255))
    ids[255 * 513:] = 7                                        # and 257 tokens of a row of another segment
    ids = ids[torch.randperm(tokens, generator=gen, device="cuda")]
    dy = torch.randn(tokens, dim, generator=gen, device="cuda")
    got = ops.embedding_backward(dy, ids, 0, rows)
    want, size = torch.zeros(rows, dim, dtype=torch.float64, device="cuda"), torch.zeros(rows, dim, dtype=torch.float64, device="cuda")
    want.index_add_(0, ids, dy.double())
    size.index_add_(0, ids, dy.double().abs())
    assert bool(((got.double() - want).abs() <= 513 * 2.0 ** -24 * size).all())
    assert torch.equal(ops.embedding_backward(dy, ids, 0, rows), got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("norm_type", [1.0, 2.0, 3.0, float("inf")])
@pytest.mark.parametrize("dim,idt", [(1, torch.int64), (7, torch.int32), (64, torch.int64), (300, torch.int32), (4100, torch.int64)])
def test_embedding_renorm_matches_oracle(ops, dtype, norm_type, dim, idt):
    """ddl_embedding_renorm on a window of a larger vocabulary, a pitched table,
    repeated ids and rows nobody looks up: looked-up rows above max_norm are
    scaled once (fp32 arithmetic, one rounding to the table's type), the others
    keep their bits."""
    gen = torch.Generator().manual_seed(dim)
    rows, lo = 40, 3
    hi = lo + rows
    store = torch.randn(rows, dim + 8, generator=gen).to(dtype)
    table = store[:, :dim]
    ids = torch.randint(0, hi + 6, (5, 13), generator=gen).to(idt)
    ids[0, :4] = lo + 7                                   # one row many times
    norms = torch.linalg.vector_norm(table.double(), ord=norm_type, dim=1)
    ordered = norms.sort().values
    max_norm = float((ordered[rows // 2 - 1] + ordered[rows // 2]) / 2)   # half of the rows are above, none is at it
    want = o_emb.renorm(table.double().numpy(), ids.numpy(), lo, hi, max_norm, norm_type)
    g_store = store.cuda()
    ops.embedding_renorm(g_store[:, :dim], ids.cuda(), lo, hi, max_norm, norm_type)
    got = g_store.cpu()
    assert torch.equal(got[:, dim:], store[:, dim:])      # the pitch is not touched
    got = got[:, :dim]
    looked_up = sorted(set(int(i) - lo for i in ids.reshape(-1).tolist() if lo <= int(i) < hi))
    scaled = [r for r in looked_up if float(norms[r]) > max_norm]
    kept = [r for r in range(rows) if r not in scaled]
    assert scaled and len(kept) > len(set(range(rows)) - set(looked_up))
    assert torch.equal(got[kept], table[kept])
    if dtype == torch.float32:
        assert np.allclose(got[scaled].double().numpy(), want[scaled], rtol=2e-6, atol=0)
    else:
        # the fp32 scale differs from the float64 one in the last bits: at most the neighbouring value of the type
        w = torch.from_numpy(want[scaled])
        near = w.to(dtype).double()
        step = (torch.nextafter(near.abs().to(dtype), torch.tensor(float("inf"), dtype=dtype)).double() - near.abs())
        assert bool(((got[scaled].double() - w).abs() <= step * 1.001).all())
    if dim > 1 or norm_type == 1.0:
        after = torch.linalg.vector_norm(got[scaled].double(), ord=norm_type, dim=1)
        assert bool((after <= max_norm * (1 + 2.0 ** -7)).all())


def test_embedding_layer_with_max_norm_matches_torch():
    """DistributedEmbedding(max_norm=...) on one worker against
    torch.nn.Embedding(max_norm=...): lookup, the table afterwards (both change
    it in place) and the gradient; on 1 x 4 workers every worker renormalises its
    own columns by their own norm (what the reference's local F.embedding call
    does), compared with the oracle per column block."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedEmbedding
    torch.manual_seed(14)
    table = torch.randn(50, 24)
    ids = torch.randint(0, 50, (3, 11))
    dy = torch.randn(3, 11, 24)
    seq = torch.nn.Embedding(50, 24, max_norm=2.5, _weight=table.clone())
    want = seq(ids)
    want.backward(dy)

    def solo(P_world):
        P_x = P_world.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1, 1])
        layer = DistributedEmbedding(P_x, 50, 24, max_norm=2.5, _weight=table.clone().cuda())
        y = layer(ids.cuda())
        y.backward(dy.cuda())
        torch.cuda.synchronize()
        return y.detach().cpu(), layer.weight.detach().cpu(), layer.weight.grad.cpu()

    y, w_after, dw = SimWorld(1).run(solo)[0]
    assert torch.allclose(y, want.detach(), rtol=1e-6, atol=1e-7)
    assert torch.allclose(w_after, seq.weight.detach(), rtol=1e-6, atol=1e-7) and not torch.equal(w_after, table)
    assert torch.allclose(dw, seq.weight.grad, rtol=1e-6, atol=1e-6)

    def body(P_world):
        P_x = P_world.create_partition_inclusive([0, 1, 2, 3]).create_cartesian_topology_partition([1, 1, 4])
        cols = slice(6 * P_x.rank, 6 * (P_x.rank + 1))
        layer = DistributedEmbedding(P_x, 50, 24, max_norm=1.2, norm_type=1.0, _weight=table[:, cols].clone().cuda())
        with torch.no_grad():
            y = layer(ids.cuda()).cpu()
        torch.cuda.synchronize()
        return y

    outs = SimWorld(4).run(body)
    for r, y in enumerate(outs):
        block = o_emb.renorm(table[:, 6 * r:6 * (r + 1)].double().numpy(), ids.numpy(), 0, 50, 1.2, 1.0)
        assert np.allclose(y.double().numpy(), o_emb.gather(block, ids.numpy(), 0, 50), rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("P,table_shape", [([1, 1], (4, 12)), ([1, 4], (4, 12)), ([1, 3], (9, 16))])
def test_embedding_training_step_reference_cases(P, table_shape):
    """The reference's test_batch_norm_with_training for the embedding
    (tests/layers/test_embedding.py:10-156; serial and 1 x 4 workers on a
    [4, 12] table, and a table whose width does not divide evenly): the table is
    scattered from one worker and handed to the layer as ``_weight``; lookup of
    every row, gather, squared-error loss, backward, a parameter step, a second
    lookup -- against torch.nn.Embedding with the reference's tolerances."""
    import math

    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedEmbedding, Repartition
    from distdl_amd.utilities.torch import zero_volume_tensor
    rtol, atol = 1e-4, math.sqrt(1e-7)
    n = int(np.prod(P))
    torch.manual_seed(0)
    table, target = torch.rand(table_shape), torch.rand(table_shape)
    ids = torch.arange(table_shape[0])
    seq = torch.nn.Embedding(*table_shape, _weight=table.clone())
    seq_out1 = seq(ids)
    seq_loss = ((seq_out1 - target) ** 2).sum()
    seq_loss.backward()
    seq_grad = seq.weight.grad.detach().clone()
    with torch.no_grad():
        seq.weight.copy_(seq.weight + 0.1 * seq.weight.grad)
        seq_out2 = seq(ids)
    want_grad = o_rep.scatter(seq_grad.numpy(), P)

    def body(P_world):
        P_root = P_world.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1])
        P_x = P_world.create_partition_inclusive(list(range(n))).create_cartesian_topology_partition(P)
        scatter, gather = Repartition(P_root, P_x), Repartition(P_x, P_root)

        def held(t):
            return t.cuda() if P_root.active else zero_volume_tensor(device="cuda")
        layer = DistributedEmbedding(P_x, *table_shape, _weight=scatter(held(table)))
        assert list(layer.P_weight.shape) == list(P)
        layer.train()
        out1 = gather(layer(ids.cuda()))
        loss = ((out1 - held(target)) ** 2).sum()
        assert loss.requires_grad
        loss.backward()
        grad = None
        if layer.P_weight.active:
            grad = layer.weight.grad.detach().cpu().numpy().copy()
            with torch.no_grad():
                layer.weight.copy_(layer.weight + 0.1 * layer.weight.grad)
        layer.eval()
        out2 = gather(layer(ids.cuda())).detach()
        torch.cuda.synchronize()
        return out1.detach().cpu(), loss.detach().cpu(), grad, out2.cpu()

    outs = SimWorld(n).run(body)
    out1, loss, _, out2 = outs[0]
    assert out1.shape == seq_out1.shape and torch.allclose(out1, seq_out1.detach(), rtol=rtol, atol=atol)
    assert torch.allclose(loss, seq_loss.detach(), rtol=rtol, atol=atol)
    assert out2.shape == seq_out2.shape and torch.allclose(out2, seq_out2, rtol=rtol, atol=atol)
    for r, (_, _, grad, _) in enumerate(outs):
        assert grad is not None and grad.shape == want_grad[r].shape
        assert np.allclose(grad, want_grad[r], rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dim,rows,tokens", [(1, 1, 1), (8, 10, 50), (100, 37, 300), (512, 64, 1000), (1000, 5, 4000),
                                              (4100, 20, 100)])
@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_embedding_backward_small_cases(ops, dtype, dim, rows, tokens, idt):
    """Window [lo, hi) of a larger vocabulary, a padding row, rows nobody looks
    up, rows looked up more than 64 times; small integers so that every sum is
    exact and the result must equal the oracle bit for bit."""
    gen = torch.Generator().manual_seed(dim + rows + tokens)
    lo, hi = 3, 3 + rows
    ids = torch.randint(0, hi + 4, (tokens,), generator=gen).to(idt)
    dy = torch.randint(-2, 3, (tokens, dim), generator=gen).to(dtype)
    pad = lo + rows // 2
    got = ops.embedding_backward(dy.cuda(), ids.cuda(), lo, hi, padding_idx=pad)
    want = o_emb.backward(dy.double().numpy(), ids.numpy(), lo, hi, padding_idx=pad)
    assert np.abs(want).max() <= 256 or dtype == torch.float32
    assert got.shape == (rows, dim) and got.dtype == dtype
    assert np.array_equal(got.cpu().double().numpy(), want)
    # no padding row, 2-D ids
    got = ops.embedding_backward(dy.cuda().reshape(1, tokens, dim), ids.cuda().reshape(1, tokens), lo, hi)
    want = o_emb.backward(dy.double().numpy(), ids.numpy(), lo, hi)
    if np.abs(want).max() <= 256 or dtype == torch.float32:
        assert np.array_equal(got.cpu().double().numpy(), want)


def test_embedding_backward_matches_torch_autograd_on_random_data(ops):
    """Random bf16 gradients: fp32 accumulation and one bf16 rounding, against
    the exact sums; and the layer-level autograd path."""
    from distdl_amd.nn.embedding import _EmbeddingShard
    gen = torch.Generator().manual_seed(12)
    table = (0.02 * torch.randn(300, 256, generator=gen)).to(torch.bfloat16)
    ids = torch.randint(0, 300, (8, 500), generator=gen)
    dy = torch.randn(8, 500, 256, generator=gen).to(torch.bfloat16)
    w = table.cuda().requires_grad_(True)
    out = _EmbeddingShard.apply(w, ids.cuda(), 0, 300, None)
    out.backward(dy.cuda())
    exact = o_emb.backward(dy.double().numpy(), ids.numpy(), 0, 300)
    got = w.grad.cpu().double().numpy()
    assert (np.abs(got - exact) <= 2.0 ** -8 * np.abs(exact) + 1e-6).all()
    # and the same through torch on the CPU in float32 (the reference's call)
    tw = table.float().requires_grad_(True)
    F.embedding(ids, tw).backward(dy.float())
    assert np.allclose(got, tw.grad.double().numpy(), rtol=2.0 ** -7, atol=1e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_embedding_backward_long_buckets_are_summed_in_token_order(ops, dtype):
    """Rows looked up 65 to several thousand times with random float gradients:
    the sums run in ascending token order whatever order the bucket fill
    produced, so the result equals a sequential fp32 sum in token order bit for
    bit, and is the same on every run.  One row exceeds what the sort holds in
    LDS (8192 tokens) and is sorted in global memory."""
    gen = torch.Generator().manual_seed(31)
    rows, dim, tokens = 12, 72, 30000
    # row 0: about 12000 tokens, row 1: about 6000, rows 2..: 65 and more, row 11: rare
    weights = torch.tensor([12000, 6000, 3000, 2000, 1500, 1200, 1000, 800, 600, 500, 300, 5], dtype=torch.float)
    ids = torch.multinomial(weights, tokens, replacement=True, generator=gen) + 4
    dy = torch.randn(tokens, dim, generator=gen).to(dtype)
    counts = torch.bincount(ids - 4, minlength=rows)
    assert int(counts[0]) > 8192 and int((counts > 64).sum()) >= 10
    first = ops.embedding_backward(dy.cuda(), ids.cuda(), 4, 4 + rows).cpu()
    want = torch.zeros(rows, dim, dtype=torch.float32)
    dy32 = dy.float()
    for r in range(rows):
        acc = torch.zeros(dim, dtype=torch.float32)
        for t in torch.nonzero(ids == r + 4).flatten().tolist():       # ascending token order, fp32, one add at a time
            acc += dy32[t]
        want[r] = acc
    assert torch.equal(first, want.to(dtype))
    for _ in range(3):
        again = ops.embedding_backward(dy.cuda(), ids.cuda(), 4, 4 + rows).cpu()
        as_bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(again.view(as_bits), first.view(as_bits))


@pytest.mark.parametrize("dtype,dim", [(torch.bfloat16, 5), (torch.bfloat16, 8), (torch.bfloat16, 255), (torch.float16, 264),
                                       (torch.bfloat16, 515), (torch.float16, 1999), (torch.float32, 3), (torch.float32, 127),
                                       (torch.float32, 129), (torch.float32, 259), (torch.float32, 770)])
@pytest.mark.parametrize("misses", [0, 150000])
def test_embedding_backward_bucket_lengths(ops, dtype, dim, misses):
    """Buckets of the lengths at which their handling changes (in registers up
    to 32 tokens, by counting up to 512, by bits per token number beyond, 1024 of
    them at a time; token numbers beyond 131072 need a second window), rows of
    whole and partial vectors and more than one group of columns, the last row of
    the table hot.  Small integers: every sum is exact in fp32, so the result is
    the exact sum rounded once."""
    lengths = [1, 2, 3, 31, 32, 33, 64, 65, 0, 511, 512, 513, 1024, 1025, 2500, 40]
    gen = torch.Generator().manual_seed(dim)
    if misses and dim > 8:
        pytest.skip("the second window does not depend on the width of the rows")
    ids = torch.cat([torch.full((n,), r) for r, n in enumerate(lengths)] + [torch.full((misses,), 99)])
    ids = ids[torch.randperm(ids.numel(), generator=gen)]
    dy = torch.randint(-1, 2, (ids.numel(), dim), generator=gen)
    got = ops.embedding_backward(dy.to(dtype).cuda(), ids.cuda(), 0, len(lengths))
    want = torch.zeros(100, dim, dtype=torch.float64).index_add_(0, ids, dy.double())[:len(lengths)]
    assert torch.equal(got.cpu(), want.to(dtype))


@pytest.mark.parametrize("rows,tokens,hot", [(1, 1, 0), (255, 1023, 40), (257, 1025, 513), (300, 1024, 1024), (5000, 20000, 4000), (5000, 20000, 4200),
                                             (2 ** 20, 70000, 600), (2 ** 20 + 1, 5000, 33), (700, 131072, 9000), (700, 131073, 9000)])
def test_embedding_backward_bucketing_by_segments(ops, rows, tokens, hot):
    """The bucketing in two launches against the four that need less workspace (but for large tables), bit for bit, and both
    against float64: one
    row and one token, a chunk of tokens and one more or less, segments with as many tokens as are held in LDS and with
    more (two hot rows share a segment), rows on either side of the lengths at which their ordering changes, table sizes
    on either side of a doubling of the segments, more tokens than one window of bits."""
    from distdl_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(rows + tokens)
    lo, pad, dim = 9, 9 + rows // 3, 5
    ids = torch.randint(0, rows + 20, (tokens,), generator=gen, device="cuda")
    where = torch.randperm(tokens, generator=gen, device="cuda")
    ids[where[:hot]] = lo + rows - 1
    ids[where[hot:hot + min(hot, 300)]] = lo + max(0, rows - 257)       # the same segment as the last row
    dy = torch.randn(tokens, dim, generator=gen, device="cuda")
    got = ops.embedding_backward(dy, ids, lo, lo + rows, padding_idx=pad)
    few = torch.full((rows, dim), 7.0, device="cuda")
    work = torch.full((3 * rows + 1 + tokens,), -1, dtype=torch.int32, device="cuda")
    assert rows >= 2 ** 20 or ops._embedding_backward_workspace(tokens, rows) > work.numel()
    rc = lib.ddl_embedding_backward(dy.data_ptr(), _lib.DDL_DT_F32, dim, dim, ids.data_ptr(), 1, tokens, lo, lo + rows, pad, 0,
                                    few.data_ptr(), dim, work.data_ptr(), work.numel(), ops._stream())
    assert rc == 0
    assert torch.equal(got.view(torch.int32), few.view(torch.int32))
    keep = (ids >= lo) & (ids < lo + rows) & (ids != pad)
    want = torch.zeros(rows, dim, dtype=torch.float64, device="cuda").index_add_(0, ids[keep] - lo, dy[keep].double())
    size = torch.zeros(rows, dim, dtype=torch.float64, device="cuda").index_add_(0, ids[keep] - lo, dy[keep].double().abs())
    count = torch.bincount(ids[keep] - lo, minlength=rows)[:, None]
    assert bool(((got.double() - want).abs() <= 2.0 ** -24 * count * size).all())    # one rounding per addition


@pytest.mark.parametrize("rows,tokens,kind", [
    (50304, 8192, "text"), (50304, 8193, "text"),          # the most tokens that one launch buckets, and one more
    (262144, 8192, "spread"), (262145, 8192, "spread"),    # the most rows of its segments, and one more
    (3, 8192, "text"), (1, 8192, "text"),                  # rows of thousands of tokens: more than a segment holds in LDS
    (700, 8192, "misses"), (256 * 20, 8184, "all hot"),    # most tokens outside of the table; every segment with a hot row
    (1000, 513, "one"), (1000, 512, "one"), (1000, 33, "one"), (1000, 32, "one"), (255, 1, "spread"), (1000, 40, "none")])
@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
def test_embedding_backward_in_one_bucketing_launch(ops, rows, tokens, kind, idt):
    """Tokens bucketed in one launch (or in two) give what the general launches give, bit for bit."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(rows + tokens)
    lo, dim = 17, 24
    if kind == "text":
        ids = (torch.exp(torch.rand(tokens, generator=gen, dtype=torch.float64) * np.log(rows + 1)).long() - 1).clamp_(0, rows - 1) + lo
    elif kind == "misses":
        ids = torch.randint(0, 20 * rows, (tokens,), generator=gen)
    elif kind == "all hot":   # 248 rows of 33 tokens each, in different segments
        ids = torch.arange(tokens)[torch.randperm(tokens, generator=gen)] % 248 + 256 * (torch.arange(1) + 19) + lo
    elif kind == "one":
        ids = torch.full((tokens,), lo + rows - 1)
    elif kind == "none":
        ids = torch.full((tokens,), lo + rows)
    else:
        ids = torch.randint(0, rows, (tokens,), generator=gen) + lo
        ids[0] = lo + rows - 1
    ids = ids.to(idt).cuda()
    dy = torch.randn(tokens, dim, generator=gen).cuda()
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    got = []
    for words in (3 * rows + 1 + tokens, max(3 * rows + 1 + tokens, lib.ddl_embedding_backward_workspace(tokens, rows))):
        work = torch.randint(-2 ** 31, 2 ** 31, (words,), generator=gen).to(torch.int32).cuda()   # whatever it held before
        dw = torch.full((rows, dim), float("nan"), device="cuda")
        _lib.check(lib.ddl_embedding_backward(dy.data_ptr(), _lib.DDL_DT_F32, dim, dim, ids.data_ptr(), int(idt == torch.int64), tokens, lo, lo + rows, lo + 5,
                                              0, dw.data_ptr(), dim, work.data_ptr(), work.numel(), stream), "ddl_embedding_backward")
        got.append(dw)
    assert torch.equal(got[0], got[1])
    assert torch.equal(ops.embedding_backward(dy, ids, lo, lo + rows, padding_idx=lo + 5), got[0])
    want = torch.zeros(rows + 1, dim, dtype=torch.float64)
    at = ids.cpu().long() - lo
    at[(at < 0) | (at >= rows) | (at == 5)] = rows
    want.index_add_(0, at, dy.cpu().double())
    # fp32 sums of up to `tokens` standard normal terms, one after the other
    most = int(torch.bincount(at, minlength=rows + 1)[:rows].max())
    assert bool(((got[0].cpu().double() - want[:rows]).abs() <= 2.0 ** -24 * most * 4 * max(most, 1) ** 0.5 + 1e-12).all())


def test_embedding_backward_of_one_row_takes_time_in_proportion_to_its_tokens(ops):
    """Every token the same id: exact sums (small integers), and four times the tokens take about four times as long (4.5
    measured; ordering the bucket anew for every 1024 of its tokens made it 22)."""
    dy = torch.randint(-3, 4, (2 ** 20, 16), device="cuda", generator=torch.Generator(device="cuda").manual_seed(20)).float()
    ids = torch.full((2 ** 20,), 7, device="cuda")
    took = []
    for n in (2 ** 18, 2 ** 20):
        times = []
        for _ in range(3):
            start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            dw = ops.embedding_backward(dy[:n], ids[:n], 0, 9)
            stop.record()
            stop.synchronize()
            times.append(start.elapsed_time(stop))
        took.append(min(times))
        want = torch.zeros(9, 16, device="cuda")
        want[7] = dy[:n].double().sum(0).float()
        assert torch.equal(dw, want)
    assert took[1] < 10 * took[0], took


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_embedding_backward_scale_grad_by_freq(ops, dtype):
    """Each row's sum divided by its number of contributing tokens, against the
    oracle (pinned to torch autograd) and through the layer's autograd path."""
    from distdl_amd.nn.embedding import _EmbeddingShard
    gen = torch.Generator().manual_seed(32)
    ids = torch.randint(0, 40, (6, 50), generator=gen)
    dy = torch.randn(6, 50, 96, generator=gen).to(dtype)
    got = ops.embedding_backward(dy.cuda(), ids.cuda(), 5, 30, padding_idx=7, scale_grad_by_freq=True)
    want = o_emb.backward(dy.double().numpy(), ids.numpy(), 5, 30, padding_idx=7, scale_grad_by_freq=True)
    tol = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 1e-5}[dtype]
    assert (np.abs(got.cpu().double().numpy() - want) <= tol * np.abs(want) + 1e-6).all()
    w = torch.zeros(25, 96, dtype=dtype, device="cuda", requires_grad=True)
    _EmbeddingShard.apply(w, ids.cuda(), 5, 30, 7, True).backward(dy.cuda())
    assert torch.equal(w.grad, got)
    plain = ops.embedding_backward(dy.cuda(), ids.cuda(), 5, 30, padding_idx=7)
    assert not torch.equal(plain, got)


def test_embedding_layer_options(ops):
    """sparse=True is refused; the id check raises on ids outside the table when switched on."""
    from distdl_amd import config
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedEmbedding

    def body(P_world):
        P_x = P_world.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1, 1])
        with pytest.raises(NotImplementedError):
            DistributedEmbedding(P_x, 10, 8, sparse=True)
        layer = DistributedEmbedding(P_x, 10, 8, scale_grad_by_freq=True)
        ids = torch.tensor([[1, 1, 1, 2]], device="cuda")
        out = layer(ids)
        out.sum().backward()
        g = layer.weight.grad.cpu()
        assert torch.allclose(g[1], torch.ones(8)) and torch.allclose(g[2], torch.ones(8)) and float(g[0].abs().sum()) == 0
        bad = torch.tensor([[1, 10]], device="cuda")
        assert float(layer(bad).detach()[0, 1].abs().sum()) == 0          # unchecked: a zero row
        config.check_embedding_ids = True
        try:
            with pytest.raises(IndexError):
                layer(bad)
            layer(ids)
        finally:
            config.check_embedding_ids = False
        return True

    assert SimWorld(1).run(body) == [True]


def test_embedding_backward_config3_rank0(ops):
    """Config 3 shapes: 131072 tokens over a 128256-row vocabulary, shard rows
    [0,16032), dim 4096 (gradient restricted to 1024 columns to keep the test
    small on the host side)."""
    gen = torch.Generator().manual_seed(1003)
    ids = torch.randint(0, 128256, (32, 4096), generator=gen)
    dy = torch.randint(-1, 2, (32, 4096, 1024), generator=gen, dtype=torch.int8).to(torch.bfloat16)
    got = ops.embedding_backward(dy.cuda(), ids.cuda(), 0, 16032)
    torch.cuda.synchronize()
    # size-independent checks: column sums over all rows equal the column sums of the hit tokens' gradients
    hit = ids < 16032
    want_total = dy[hit].double().sum(0)
    assert torch.equal(got.cpu().double().sum(0), want_total)
    # rows never looked up are zero, a sample of rows is exact
    looked = torch.zeros(16032, dtype=torch.bool)
    looked[ids[hit]] = True
    assert int((got.cpu()[~looked] != 0).sum()) == 0
    sample = torch.nonzero(looked).flatten()[:64]
    for r in sample.tolist():
        assert torch.equal(got[r].cpu().double(), dy[ids == r].double().sum(0))


# ------------------------------------------------------------------- Linear --

def _lin_check(got_bits, x, w, b, sample_rows=None):
    xb, wb = bits16(x), bits16(w)
    bb = None if b is None else bits16(b)
    if sample_rows is not None:
        xb = xb.reshape(-1, xb.shape[-1])[sample_rows]
        got_bits = got_bits.reshape(-1, got_bits.shape[-1])[sample_rows]
    exact = o_lin.linear(xb, wb, bb, dtype=np.float64)
    got = o_lin.bf16_bits_to_f32(got_bits).astype(np.float64).reshape(exact.shape)
    k = x.shape[-1]
    # |error| <= rtol * (|exact| + typical magnitude of the K-term sum): rounding to bf16 is 2^-9 relative,
    # fp32 accumulation error is far below; cancellation in the sum is covered by the magnitude term
    mag = np.sqrt(k) * float(x.float().abs().mean()) * float(w.float().abs().mean()) + 1e-30
    err = np.abs(got - exact)
    assert (err <= LIN_RTOL * (np.abs(exact) + mag)).all(), float((err / (np.abs(exact) + mag)).max())
    # tighter, aggregate: relative Frobenius error is at bf16 rounding level
    assert np.linalg.norm(got - exact) <= 4e-3 * np.linalg.norm(exact) + 1e-30


@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (32, 32, 16), (256, 256, 64), (300, 200, 72), (513, 259, 136),
                                   (64, 1000, 4096), (1024, 512, 512)])
@pytest.mark.parametrize("use_bias", [True, False])
def test_linear_small_integer_cases_are_exact(ops, M, N, K, use_bias):
    """Small integers: every product and partial sum is exact in fp32, results
    are below 2^8 so bf16 holds them exactly when |y| <= 256 -- any indexing
    mistake in the tiling shows as a wrong integer."""
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    x = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16)
    w = torch.randint(-1, 2, (N, K), generator=gen).to(torch.bfloat16)
    # keep |y| small: zero most of each weight row
    mask = (torch.rand(N, K, generator=gen) < (64.0 / K)).to(torch.bfloat16)
    w = w * mask
    b = torch.randint(-3, 4, (N,), generator=gen).to(torch.bfloat16) if use_bias else None
    y = ops.linear_bf16(x.cuda(), w.cuda(), None if b is None else b.cuda())
    want = x.double() @ w.double().T
    if b is not None:
        want = want + b.double()
    assert want.abs().max() <= 256
    assert torch.equal(y.cpu().double(), want)


@pytest.mark.parametrize("M,N,K,ldy", [(300, 259, 72, 264), (513, 100, 136, 104), (70, 255, 64, 512), (257, 36, 32, 36)])
def test_linear_strided_output_through_the_c_abi(ops, M, N, K, ldy):
    """Output rows with a pitch larger than N (and N not a multiple of the
    16-byte store width): results exact, the gap between rows untouched."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M + 3 * N + K)
    x = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16)
    w = torch.randint(-1, 2, (N, K), generator=gen).to(torch.bfloat16)
    b = torch.randint(-3, 4, (N,), generator=gen).to(torch.bfloat16)
    xg, wg, bg = x.cuda(), w.cuda(), b.cuda()
    out = torch.full((M, ldy), 77.0, dtype=torch.bfloat16, device="cuda")
    rc = _lib.load().ddl_linear_bf16(xg.data_ptr(), wg.data_ptr(), bg.data_ptr(), out.data_ptr(), M, N, K, K, K, ldy,
                                     torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ddl_linear_bf16")
    want = x.double() @ w.double().T + b.double()
    assert want.abs().max() <= 256
    got = out.cpu().double()
    assert torch.equal(got[:, :N], want)
    assert (got[:, N:] == 77.0).all()


@pytest.mark.parametrize("M,N,K", [(128, 96, 256), (777, 333, 1024), (2048, 1024, 512)])
def test_linear_random_within_tolerance(ops, M, N, K):
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, generator=gen)).to(torch.bfloat16)
    b = (0.02 * torch.randn(N, generator=gen)).to(torch.bfloat16)
    y = ops.linear_bf16(x.cuda(), w.cuda(), b.cuda())
    _lin_check(bits16(y), x, w, b)
    # the reference's call on the same bits, on the CPU
    ref = F.linear(x.float(), w.float(), b.float())
    assert torch.allclose(y.cpu().float(), ref, rtol=LIN_RTOL, atol=LIN_RTOL * float(ref.abs().mean()))


def test_linear_config4_rank0(ops):
    """x [4,2048,8192] ~ N(0,1); weight shard [3584,8192] ~ N(0,0.02); bias [3584]."""
    gen = torch.Generator().manual_seed(1004)
    x = torch.randn(4, 2048, 8192, generator=gen).to(torch.bfloat16)
    w = (0.02 * torch.randn(3584, 8192, generator=gen)).to(torch.bfloat16)
    b = (0.02 * torch.randn(3584, generator=gen)).to(torch.bfloat16)
    xg, wg, bg = x.cuda(), w.cuda(), b.cuda()
    y = ops.linear_bf16(xg, wg, bg)
    torch.cuda.synchronize()
    assert y.shape == (4, 2048, 3584)
    rows = np.r_[0:64, 255:258, 4090:4100, 8128:8192]           # tile borders and both ends
    _lin_check(bits16(y), x, w, b, sample_rows=rows)
    # size-independent property on the whole output: linearity in x.
    # y(2x) - bias == 2 (y(x) - bias) exactly up to the final bf16 rounding
    y2 = ops.linear_bf16((2 * xg), wg, None)
    y1 = ops.linear_bf16(xg, wg, None)
    assert torch.equal(y2, 2 * y1)
    # and agreement of every element with the same GEMM evaluated by rocBLAS in fp32
    ref = (xg.float().reshape(-1, 8192) @ wg.float().T + bg.float()).reshape(4, 2048, 3584)
    rel = (y.float() - ref).abs() / (ref.abs() + 0.02 * np.sqrt(8192) * 0.8)
    assert float(rel.max()) <= LIN_RTOL


@pytest.mark.parametrize("rows,cols", [(1, 1), (64, 64), (65, 63), (300, 130), (1000, 8), (7, 513)])
def test_transpose_2d_is_bit_exact(ops, rows, cols):
    gen = torch.Generator().manual_seed(rows * 1000 + cols)
    src = torch.randint(-32768, 32767, (rows, cols), generator=gen, dtype=torch.int16)
    got = ops.transpose_2d(src.cuda())
    assert torch.equal(got.cpu(), src.t().contiguous())
    # padded pitch: the extra columns are zero
    ld = (rows + 7) // 8 * 8 + 8
    got = ops.transpose_2d(src.cuda(), ld)
    assert torch.equal(got[:, :rows].cpu(), src.t().contiguous()) and (got[:, rows:] == 0).all()
    # a strided source view
    wide = torch.randint(-32768, 32767, (rows, cols + 5), generator=gen, dtype=torch.int16).cuda()
    assert torch.equal(ops.transpose_2d(wide[:, 2:2 + cols]).cpu(), wide[:, 2:2 + cols].cpu().t().contiguous())


@pytest.mark.parametrize("rows,cols", [(1, 1), (8, 8), (63, 65), (64, 64), (65, 127), (515, 9), (7, 1025)])
@pytest.mark.parametrize("address,pitch", [(0, 0), (1, 1), (3, 6)])
def test_padded_transpose_and_padded_rows_at_any_address(ops, rows, cols, address, pitch):
    """Every bit arrives, the padding is cleared whatever was there, and nothing past it is touched; rows at any 2-byte
    address and pitch, also one row read again and again."""
    from distdl_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(rows * 100 + cols)
    ld = cols + pitch
    pool = torch.randint(-32768, 32767, (rows * ld + address,), generator=gen, dtype=torch.int16)
    src = pool[address:].view(rows, ld)[:, :cols]
    dev = pool.cuda()
    ptr = dev.data_ptr() + 2 * address
    width = (rows + 7) // 8 * 8
    for more, start in ((0, 0), (5, 0), (3, 1)):              # columns of dst past the padding; its address in elements
        dst = torch.full((cols * (width + more) + start + 8,), 77, dtype=torch.int16, device="cuda")
        _lib.check(lib.ddl_transpose_padded(ptr, dst.data_ptr() + 2 * start, rows, cols, ld, width + more, width, 2, None), "t")
        got = dst.cpu()
        body = got[start:start + cols * (width + more)].view(cols, width + more)
        assert torch.equal(body[:, :rows], src.t()) and not body[:, rows:width].any() and (body[:, width:] == 77).all()
        assert (got[:start] == 77).all() and (got[-8:] == 77).all()
    width = (cols + 7) // 8 * 8 + 8
    for step in (ld, 0):
        dst = torch.full((rows * width + 8,), 77, dtype=torch.int16, device="cuda")
        _lib.check(lib.ddl_pad_rows(ptr, dst.data_ptr(), rows, cols, step, width, 2, None), "p")
        got = dst.cpu()
        body = got[:rows * width].view(rows, width)
        assert torch.equal(body[:, :cols], src if step else src[:1].expand(rows, cols))
        assert not body[:, cols:].any() and (got[-8:] == 77).all()
    assert lib.ddl_transpose_padded(ptr, dst.data_ptr(), rows, cols, ld, rows, rows + 1, 2, None) == -1
    assert lib.ddl_pad_rows(ptr, dst.data_ptr(), rows, cols, ld, cols + 7 - (cols + 6) % 8, 2, None) == -1


@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 3), (128, 64), (129, 65), (8192, 200), (3000, 1000)])
def test_colsum_bf16(ops, rows, cols):
    gen = torch.Generator().manual_seed(rows + cols)
    a = torch.randn(rows, cols, generator=gen).to(torch.bfloat16)
    got = ops.colsum_bf16(a.cuda()).cpu().double()
    exact = a.double().sum(0)
    # fp32 accumulation of bf16 values, one bf16 rounding of the result
    tol = 2.0 ** -8 * exact.abs() + 1e-5 * a.double().abs().sum(0)
    assert ((got - exact).abs() <= tol).all()
    # small integers: exact
    ai = torch.randint(-2, 3, (rows, cols), generator=gen).to(torch.bfloat16)
    want = ai.double().sum(0)
    if want.abs().max() <= 256:
        assert torch.equal(ops.colsum_bf16(ai.cuda()).cpu().double(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols,pad", [(1, 1, 0), (3, 3, 2), (70, 5, 0), (513, 7, 0), (600, 8, 1), (64, 9, 0), (1000, 15, 0), (1025, 16, 3), (33, 17, 0),
                                           (777, 333, 0), (4096, 143, 5), (4097, 143, 5), (2100, 70, 1), (129, 4103, 0)])
def test_colsum_of_rows_at_any_address(ops, dtype, rows, cols, pad):
    """Rows of odd length and pitch that start one element into their buffer and end where it ends, in one launch and in two;
    columns whose last vector starts inside the one before it, rows shorter than a vector.  NaN lies between the rows.  Small
    integers: the sums are exact."""
    a = torch.randint(-2, 3, (rows, cols), generator=torch.Generator().manual_seed(rows + cols)).to(dtype)
    store = torch.full((1 + rows * (cols + pad) - pad,), float("nan"), dtype=dtype, device="cuda")
    ag = store[1:].as_strided((rows, cols), (cols + pad, 1), 1)
    ag.copy_(a)
    assert torch.equal(ops.colsum(ag).cpu(), a.double().sum(0).to(dtype))


@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (96, 80, 128), (300, 200, 72), (257, 36, 40), (5, 3, 16), (64, 1000, 256)])
def test_linear_backward_small_integer_cases_are_exact(ops, M, N, K):
    """dx = dy w, dw = dy^T x, db = sum dy with small integers: every sum is
    exact in fp32 and representable in bf16, so the results must be the exact
    integers -- a wrong transpose or pitch shows at once."""
    gen = torch.Generator().manual_seed(M * 5 + N * 3 + K)
    x = torch.randint(-1, 2, (M, K), generator=gen).to(torch.bfloat16)
    w = torch.randint(-1, 2, (N, K), generator=gen).to(torch.bfloat16)
    dy = torch.randint(-1, 2, (M, N), generator=gen).to(torch.bfloat16)
    # keep the sums below 2^8: thin out dy and w
    dy = dy * (torch.rand(M, N, generator=gen) < min(1.0, 40.0 / max(M, N))).to(torch.bfloat16)
    w = w * (torch.rand(N, K, generator=gen) < min(1.0, 40.0 / N)).to(torch.bfloat16)
    dx, dw, db = ops.linear_bf16_backward(x.cuda(), w.cuda(), dy.cuda())
    want_dx, want_dw, want_db = o_lin.linear_backward(bits16(x), bits16(w), bits16(dy))
    assert max(np.abs(want_dx).max(), np.abs(want_dw).max(), np.abs(want_db).max()) <= 256
    assert np.array_equal(dx.cpu().double().numpy(), want_dx)
    assert np.array_equal(dw.cpu().double().numpy(), want_dw)
    assert np.array_equal(db.cpu().double().numpy(), want_db)


def test_linear_backward_config4_rank0(ops):
    """The adjoint of configuration 4 at its full size (M 8192, N 3584, K 8192):
    dx = dy w [8192, 8192], dw = dy^T x [3584, 8192], db = column sums, on the
    operands where they lie.  Sampled rows (tile borders and both ends) against
    the oracle's exact sums; on the whole outputs, linearity in dy (a factor of
    two is exact in bf16) and agreement with the same products by the vendor
    GEMM in fp32."""
    gen = torch.Generator().manual_seed(1404)
    x = torch.randn(8192, 8192, generator=gen).to(torch.bfloat16)
    w = (0.02 * torch.randn(3584, 8192, generator=gen)).to(torch.bfloat16)
    dy = torch.randn(8192, 3584, generator=gen).to(torch.bfloat16)
    xg, wg, dyg = x.cuda(), w.cuda(), dy.cuda()
    dx, dw, db = ops.linear_bf16_backward(xg, wg, dyg)
    torch.cuda.synchronize()
    assert dx.shape == (8192, 8192) and dw.shape == (3584, 8192) and db.shape == (3584,)
    xb, wb, dyb = bits16(x), bits16(w), bits16(dy)
    rows = np.r_[0:16, 255:258, 4094:4098, 8176:8192]
    want_dx = o_lin.bf16_bits_to_f32(dyb[rows]).astype(np.float64) @ o_lin.bf16_bits_to_f32(wb).astype(np.float64)
    err = np.abs(dx[rows].cpu().double().numpy() - want_dx)
    assert (err <= LIN_RTOL * (np.abs(want_dx) + np.abs(want_dx).mean())).all()
    nrows = np.r_[0:16, 191:194, 2046:2050, 3568:3584]
    want_dw = o_lin.bf16_bits_to_f32(dyb[:, nrows]).astype(np.float64).T @ o_lin.bf16_bits_to_f32(xb).astype(np.float64)
    err = np.abs(dw[nrows].cpu().double().numpy() - want_dw)
    assert (err <= LIN_RTOL * (np.abs(want_dw) + np.abs(want_dw).mean())).all()
    want_db = o_lin.bf16_bits_to_f32(dyb).astype(np.float64).sum(axis=0)
    err = np.abs(db.cpu().double().numpy() - want_db)
    assert (err <= LIN_RTOL * (np.abs(want_db) + np.abs(want_db).mean())).all()
    dx2, dw2, db2 = ops.linear_bf16_backward(xg, wg, 2 * dyg)
    assert torch.equal(dx2, 2 * dx) and torch.equal(dw2, 2 * dw) and torch.equal(db2, 2 * db)
    ref_dx = dyg.float() @ wg.float()
    assert float(((dx.float() - ref_dx).abs() / (ref_dx.abs() + ref_dx.abs().mean())).max()) <= LIN_RTOL
    del ref_dx
    ref_dw = dyg.float().t() @ xg.float()
    assert float(((dw.float() - ref_dw).abs() / (ref_dw.abs() + ref_dw.abs().mean())).max()) <= LIN_RTOL


def test_layernorm_backward_config1_rank0(ops):
    """The adjoint of configuration 1 at its full size: rank 0's shard
    [8192, 256] of rows of 1024 over four workers, the other workers' row sums
    seeded from the oracle's fp64 quantities.  dx, dgamma, dbeta of both the
    two-launch and the one-pass form against the fp64 closed form."""
    rng = np.random.default_rng(1401)
    rows, cols, P, eps = 16 * 512, 256, 4, 1e-5
    xg = rng.standard_normal((rows, P * cols)).astype(np.float32)
    dyg = rng.standard_normal((rows, P * cols)).astype(np.float32)
    gamma = (1 + 0.1 * rng.standard_normal(P * cols)).astype(np.float32)
    shards = [np.ascontiguousarray(xg[:, cols * p:cols * (p + 1)]) for p in range(P)]
    dys = [np.ascontiguousarray(dyg[:, cols * p:cols * (p + 1)]) for p in range(P)]
    gammas = [gamma[cols * p:cols * (p + 1)] for p in range(P)]
    want_dx, want_dg, want_db = o_ln.backward_shards(shards, gammas, dys, eps)
    x2d, dy2d, g = torch.from_numpy(shards[0]).cuda(), torch.from_numpy(dys[0]).cuda(), torch.from_numpy(gammas[0]).cuda()
    parts = [torch.from_numpy(o_ln.partial_stats(s).astype(np.float32)).cuda() for s in shards]
    parts[0] = ops.ln_partial_stats(x2d)
    beta = torch.zeros(cols, device="cuda")
    _, mean, rstd = ops.ln_normalize_affine(x2d, torch.stack(parts).contiguous(), [cols] * P, g, beta, eps, want_stats=True)
    m64 = xg.astype(np.float64).mean(axis=1)
    r64 = 1.0 / np.sqrt(xg.astype(np.float64).var(axis=1) + eps)
    gathered = []
    for p in range(P):
        gp = dys[p].astype(np.float64) * gammas[p].astype(np.float64)
        xh = (shards[p].astype(np.float64) - m64[:, None]) * r64[:, None]
        gathered.append(torch.from_numpy(np.stack([gp.sum(axis=1), (gp * xh).sum(axis=1)], axis=1).astype(np.float32)).cuda())
    sums, work = ops.ln_backward_partial_params(dy2d, x2d, mean, rstd, g)
    assert np.allclose(sums.cpu().numpy(), gathered[0].cpu().numpy(), rtol=1e-4, atol=1e-3)
    gathered[0] = sums
    table = torch.stack(gathered).contiguous()
    dx, dg, db = ops.ln_backward_input_params(dy2d, x2d, mean, rstd, g, table, 1.0 / (P * cols), work)
    torch.cuda.synchronize()
    tol = 1e-5 * max(1.0, np.abs(want_dx[0]).max())
    assert np.abs(dx.cpu().numpy() - want_dx[0]).max() <= 4 * tol
    # column sums over 8192 rows of O(1) terms: 1e-5 of the sum of magnitudes
    assert np.abs(dg.cpu().numpy() - want_dg[0]).max() <= 1e-5 * np.abs(dys[0]).sum(axis=0).max() * 4
    assert np.abs(db.cpu().numpy() - want_db[0]).max() <= 1e-5 * np.abs(dys[0]).sum(axis=0).max()
    poisoned = table.clone()
    poisoned[0] = float("nan")
    dx1, dg1, db1 = ops.ln_backward_one_pass(dy2d, x2d, mean, rstd, g, 1.0 / (P * cols), poisoned, 0)
    torch.cuda.synchronize()
    assert torch.equal(poisoned, table) and torch.equal(dx1, dx) and torch.equal(dg1, dg) and torch.equal(db1, db)


def test_linear_shard_autograd_matches_torch(ops):
    """The reference's layer runs torch autograd through F.linear; the same
    gradients must come out of the HIP path (bf16 tolerance), including through
    a batch-shaped input and with no bias."""
    from distdl_amd.nn.linear import linear_shard
    gen = torch.Generator().manual_seed(9)
    x = torch.randn(3, 50, 96, generator=gen).to(torch.bfloat16)
    w = (0.05 * torch.randn(72, 96, generator=gen)).to(torch.bfloat16)
    b = (0.05 * torch.randn(72, generator=gen)).to(torch.bfloat16)
    dy = torch.randn(3, 50, 72, generator=gen).to(torch.bfloat16)
    for use_bias in (True, False):
        xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
        bg = b.cuda().requires_grad_(True) if use_bias else None
        linear_shard(xg, wg, bg).backward(dy.cuda())
        xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
        br = b.double().requires_grad_(True) if use_bias else None
        F.linear(xr, wr, br).backward(dy.double())
        for got, ref in ((xg.grad, xr.grad), (wg.grad, wr.grad)) + (((bg.grad, br.grad),) if use_bias else ()):
            assert got.dtype == torch.bfloat16 and got.shape == ref.shape
            err = (got.cpu().double() - ref).abs()
            assert (err <= LIN_RTOL * (ref.abs() + ref.abs().mean())).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (32, 32, 16), (300, 200, 72), (513, 259, 136), (130, 1000, 1024), (7, 5, 3),
                                   (129, 131, 17)])
@pytest.mark.parametrize("use_bias", [True, False])
def test_linear_fp16_and_fp32_small_integer_cases_are_exact(ops, dtype, M, N, K, use_bias):
    """Small integers: every product and partial sum is exact, so the result
    must equal the fp64 product exactly -- any indexing mistake shows.  fp32
    takes any K; fp16 shapes with K not a multiple of 8 go through the padded
    copies."""
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    x = torch.randint(-2, 3, (M, K), generator=gen).to(dtype)
    w = torch.randint(-2, 3, (N, K), generator=gen).to(dtype)
    b = torch.randint(-3, 4, (N,), generator=gen).to(dtype) if use_bias else None
    y = ops.linear(x.cuda(), w.cuda(), None if b is None else b.cuda())
    want = x.double() @ w.double().T + (0 if b is None else b.double())
    assert y.dtype == dtype and y.shape == (M, N)
    assert torch.equal(y.cpu().double(), want)


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2.0 ** -9), (torch.float32, 1e-5)])
def test_linear_fp16_and_fp32_random_within_tolerance(ops, dtype, tol):
    """Random operands against the fp64 product of the same values: fp32
    accumulation and one rounding to the result type."""
    gen = torch.Generator().manual_seed(77)
    M, N, K = 384, 520, 2048
    x = torch.randn(3, M // 3, K, generator=gen).to(dtype)
    w = (0.05 * torch.randn(N, K, generator=gen)).to(dtype)
    b = torch.randn(N, generator=gen).to(dtype)
    y = ops.linear(x.cuda(), w.cuda(), b.cuda())
    exact = x.double().reshape(-1, K) @ w.double().T + b.double()
    mag = np.sqrt(K) * float(x.float().abs().mean()) * float(w.float().abs().mean())
    err = (y.cpu().double().reshape(-1, N) - exact).abs()
    assert bool((err <= tol * (exact.abs() + mag) + 1e-30).all()), float((err / (exact.abs() + mag)).max())
    # the reference's call on the same values, on the CPU in float32
    ref = F.linear(x.float(), w.float(), b.float())
    assert torch.allclose(y.cpu().float(), ref, rtol=4 * tol, atol=4 * tol * float(ref.abs().mean()))


def test_linear_bf16_forward_pads_unaligned_operands(ops):
    """K not a multiple of 8, an offset view as input: the layer-level entry
    copies into padded temporaries instead of refusing (the C entry point refuses)."""
    gen = torch.Generator().manual_seed(5)
    for K in (1, 12, 33):
        x = torch.randint(-2, 3, (40, K), generator=gen).to(torch.bfloat16)
        w = torch.randint(-2, 3, (24, K), generator=gen).to(torch.bfloat16)
        y = ops.linear(x.cuda(), w.cuda())
        assert torch.equal(y.cpu().double(), x.double() @ w.double().T)
    base = torch.randint(-2, 3, (50, 72), generator=gen).to(torch.bfloat16).cuda()
    view = base[3:43, 4:68]                                    # pitch 72, first element 8 bytes off a 16-byte boundary
    w = torch.randint(-2, 3, (16, 64), generator=gen).to(torch.bfloat16)
    y = ops.linear(view, w.cuda())
    assert torch.equal(y.cpu().double(), view.cpu().double() @ w.double().T)
    from distdl_amd import _lib
    rc = _lib.load().ddl_linear(view.data_ptr(), w.cuda().data_ptr(), None, y.data_ptr(), _lib.DDL_DT_BF16, 40, 16, 64, 72, 64, 16,
                                None)
    assert rc == -3


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 48, 40), (300, 130, 72), (5, 3, 2), (129, 257, 33)])
def test_linear_backward_fp16_and_fp32_exact_and_autograd(ops, dtype, M, N, K):
    """dx = dy w, dw = dy^T x, db = column sums on small integers (exact), and
    the autograd hook-up of the shard against torch's on the CPU."""
    from distdl_amd.nn.linear import linear_shard
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randint(-2, 3, (M, K), generator=gen).to(dtype)
    w = torch.randint(-2, 3, (N, K), generator=gen).to(dtype)
    dy = torch.randint(-2, 3, (M, N), generator=gen).to(dtype)
    dx, dw, db = ops.linear_backward(x.cuda(), w.cuda(), dy.cuda())
    assert torch.equal(dx.cpu().double(), dy.double() @ w.double())
    assert torch.equal(dw.cpu().double(), dy.double().T @ x.double())
    assert torch.equal(db.cpu().double(), dy.double().sum(0))
    xg, wg = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    bg = torch.zeros(N, dtype=dtype, device="cuda", requires_grad=True)
    linear_shard(xg, wg, bg).backward(dy.cuda())
    xr, wr, br = x.double().requires_grad_(True), w.double().requires_grad_(True), torch.zeros(N, dtype=torch.double, requires_grad=True)
    F.linear(xr, wr, br).backward(dy.double())
    assert torch.equal(xg.grad.cpu().double(), xr.grad) and torch.equal(wg.grad.cpu().double(), wr.grad)
    assert torch.equal(bg.grad.cpu().double(), br.grad)


def test_linear_layers_run_in_float32_like_the_reference_tests(ops):
    """DistributedLinear keeps torch's default dtype, as in the reference's
    layer tests (tests/layers/test_linear.py:48-305 build float32 layers): the
    shard runs on the fp32 kernel, forward and backward, against torch on the CPU."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLinear, DistributedLinearAllGather
    Pw = SimWorld(8).partition(0)
    P_x = Pw.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1])
    P_y = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([1, 8])
    P_w = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([8, 1])
    torch.manual_seed(9)
    layer = DistributedLinear(P_x, P_y, P_w, 60, 400)
    assert layer.sublinear.weight.dtype == torch.float32 and tuple(layer.sublinear.weight.shape) == (50, 60)
    x = torch.randn(33, 60)
    xg = x.cuda().requires_grad_(True)
    y = layer(xg)
    y.backward(torch.ones_like(y))
    w, b = layer.sublinear.weight.detach().cpu(), layer.sublinear.bias.detach().cpu()
    xr = x.clone().requires_grad_(True)
    wr, br = w.clone().requires_grad_(True), b.clone().requires_grad_(True)
    yr = F.linear(xr, wr, br)
    yr.backward(torch.ones_like(yr))
    assert torch.allclose(y.detach().cpu(), yr.detach(), rtol=1e-5, atol=1e-5)
    assert torch.allclose(xg.grad.cpu(), xr.grad, rtol=1e-5, atol=1e-5)
    assert torch.allclose(layer.sublinear.weight.grad.cpu(), wr.grad, rtol=1e-5, atol=1e-4)
    assert torch.allclose(layer.sublinear.bias.grad.cpu(), br.grad, rtol=1e-5, atol=1e-5)
    P_y3 = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([1, 1, 8])
    ag = DistributedLinearAllGather(P_y3, 72, 160)
    assert ag.weight.dtype == torch.float32
    x3 = torch.randn(2, 9, 72)
    with torch.no_grad():
        y3 = ag(x3.cuda())
    want = F.linear(x3, ag.weight.detach().cpu().view(20, 72), ag.bias.detach().cpu().view(20))
    assert torch.allclose(y3.cpu(), want, rtol=1e-5, atol=1e-5)


def _gemm_operand(values, transposed, pad):
    """Device tensor holding ``values[rows, k]`` contiguous along k, or (transposed)
    along the rows, with `pad` unused elements at the end of each line; returns
    (tensor, row_stride, k_stride)."""
    rows, k = values.shape
    if transposed:
        store = torch.full((k, rows + pad), 3.0, dtype=values.dtype)
        store[:, :rows] = values.T
        return store.cuda(), 1, rows + pad
    store = torch.full((rows, k + pad), 3.0, dtype=values.dtype)
    store[:, :k] = values
    return store.cuda(), k + pad, 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,pad", [(8, 8, 8, 0), (16, 24, 72, 8), (304, 200, 136, 0), (264, 40, 64, 16), (520, 776, 200, 8),
                                       (4096, 4352, 136, 0), (64, 192, 4104, 0), (4096, 4096, 72, 0), (8192, 3592, 72, 8)])
def test_gemm_16_bit_reads_operands_where_they_lie(ops, dtype, a_t, b_t, M, N, K, pad):
    """ddl_gemm on every combination of operand layouts (contiguous along k or
    along the rows), with small integers so that the result must be the exact
    integer: tiles that straddle M, N and K, pitched operands, one k-tile and
    many; products small enough for the 128-row tiles, one that fills the chip
    with 256 x 256 tiles, and one that is split between wide and narrow tiles."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K + 2 * a_t + b_t)
    a = torch.randint(-1, 2, (M, K), generator=gen).to(dtype)
    b = torch.randint(-1, 2, (N, K), generator=gen).to(dtype)
    b = b * (torch.rand(N, K, generator=gen) < min(1.0, 64.0 / K)).to(dtype)
    bias = torch.randint(-3, 4, (N,), generator=gen).to(dtype)
    ag, a_rs, a_ks = _gemm_operand(a, a_t, pad)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, pad)
    ldy = N + 8
    out = torch.full((M, ldy), 77.0, dtype=dtype, device="cuda")
    dt = _lib.DDL_DT_BF16 if dtype == torch.bfloat16 else _lib.DDL_DT_F16
    rc = _lib.load().ddl_gemm(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, bias.cuda().data_ptr(), out.data_ptr(), dt, ldy,
                              M, N, K, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ddl_gemm")
    want = a.double() @ b.double().T + bias.double()
    assert want.abs().max() <= 256
    got = out.cpu().double()
    assert torch.equal(got[:, :N], want)
    assert (got[:, N:] == 77.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_t,b_t,M,N,K,splits", [
    # up to 64 rows: one to eight pieces of eight rows, odd columns, one step per wavefront and many, a straddling step
    (False, False, 1, 1, 8, False), (False, False, 8, 17, 512, False), (False, False, 9, 40, 1032, False),
    (False, False, 17, 333, 4104, False), (False, False, 33, 16, 520, False), (False, False, 64, 100, 2056, False),
    # small tiles: one workgroup and several per CU, one k-tile and an odd number of them
    (False, False, 65, 65, 64, False), (False, True, 72, 136, 200, False), (True, False, 136, 67, 456, False),
    (True, True, 2056, 1032, 136, False),
    # the reduction split over workgroups: unequal shares, a share that straddles K
    (False, False, 100, 130, 4168, True), (False, True, 72, 136, 4168, True), (True, False, 200, 264, 4104, True),
    (True, True, 128, 64, 8191, True)])
def test_gemm_16_bit_products_that_leave_the_chip_idle(ops, dtype, a_t, b_t, M, N, K, splits):
    """The skinny and small-tile kernels on integer operands (every sum is exact), with and without the workspace that
    lets them split the reduction; the workspace's contents on entry do not matter."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    a = torch.randint(-1, 2, (M, K), generator=gen).to(dtype)
    b = torch.randint(-1, 2, (N, K), generator=gen).to(dtype)
    b = b * (torch.rand(N, K, generator=gen) < min(1.0, 64.0 / K)).to(dtype)
    bias = torch.randint(-3, 4, (N,), generator=gen).to(dtype)
    ag, a_rs, a_ks = _gemm_operand(a, a_t, 0)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, 0)
    want = a.double() @ b.double().T + bias.double()
    assert want.abs().max() <= 256
    lib, dt, stream = _lib.load(), _lib.DDL_DT_BF16 if dtype == torch.bfloat16 else _lib.DDL_DT_F16, torch.cuda.current_stream().cuda_stream
    elems = lib.ddl_gemm_workspace(dt, a_rs, a_ks, b_rs, b_ks, M, N, K)
    assert (elems > 0) == splits
    ldy = N + 8
    for n in {0, elems // 2, elems}:
        work = torch.full((n,), float("nan"), device="cuda") if n else None
        out = torch.full((M, ldy), 77.0, dtype=dtype, device="cuda")
        rc = lib.ddl_gemm_ws(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, bias.cuda().data_ptr(), out.data_ptr(), dt, ldy, M, N,
                             K, None if work is None else work.data_ptr(), n, stream)
        _lib.check(rc, "ddl_gemm_ws")
        got = out.cpu().double()
        assert torch.equal(got[:, :N], want)
        assert (got[:, N:] == 77.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,pad", [
    # every operand shape whose pitch, length or address is no multiple of eight: one k-tile that straddles K, whole k-tiles, an
    # odd number of them, a reduction split over workgroups; tiles that straddle M and N by one and by seven
    (8, 8, 1, 0), (9, 11, 3, 1), (65, 63, 65, 0), (71, 137, 640, 3), (201, 263, 1033, 0), (1030, 1023, 127, 0), (15, 66, 8191, 2)])
def test_gemm_16_bit_operands_at_any_pitch(ops, dtype, a_t, b_t, M, N, K, pad):
    """The kernel for unaligned 16-bit operands on integers (every sum is exact), read where they lie and against the
    refusal of the aligned entry point; the operands end where their buffers end."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M * 7 + N * 3 + K + 2 * a_t + b_t)
    a = torch.randint(-1, 2, (M, K), generator=gen).to(dtype)
    b = torch.randint(-1, 2, (N, K), generator=gen).to(dtype)
    b = b * (torch.rand(N, K, generator=gen) < min(1.0, 64.0 / K)).to(dtype)
    bias = torch.randint(-3, 4, (N,), generator=gen).to(dtype)
    ag, a_rs, a_ks = _gemm_operand(a, a_t, pad)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, pad)
    shift_a = torch.empty(ag.numel() + 1, dtype=dtype, device="cuda")      # the same operand one element further on
    shift_a[1:] = ag.reshape(-1)
    lib, dt, stream = _lib.load(), _lib.DDL_DT_BF16 if dtype == torch.bfloat16 else _lib.DDL_DT_F16, torch.cuda.current_stream().cuda_stream
    want = a.double() @ b.double().T + bias.double()
    assert want.abs().max() <= 256
    elems = max(1 << 20, lib.ddl_gemm_workspace(dt, a_rs, a_ks, b_rs, b_ks, M, N, K))
    assert lib.ddl_gemm_in_place(dt, 0, a_rs, a_ks, b_rs, b_ks, M, N, K) == 1
    work, ldy = torch.full((elems,), float("nan"), device="cuda"), N + 3
    for ptr in (ag.data_ptr(), shift_a.data_ptr() + 2):
        out = torch.full((M, ldy), 77.0, dtype=dtype, device="cuda")
        args = (ptr, a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, bias.cuda().data_ptr(), out.data_ptr(), dt, ldy, M, N, K)
        if ptr % 16:
            assert lib.ddl_gemm(*args, stream) == -3
        _lib.check(lib.ddl_gemm_ws(*args, work.data_ptr(), elems, stream), "ddl_gemm_ws")
        got = out.cpu().double()
        assert torch.equal(got[:, :N], want)
        assert (got[:, N:] == 77.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(8, 64, 32768), (2, 128, 28672), (1, 8, 57344), (8, 3584, 8192), (64, 256, 4096)])
def test_linear_of_operands_off_a_16_byte_boundary(ops, dtype, M, N, K):
    """x one element into its buffer, pitches that are multiples of eight: the product and its adjoint through the front end,
    which sizes the workspace, and the product with that workspace, half of it and none.  Integers, every sum is exact."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randint(-1, 2, (M, K), generator=gen).to(dtype)
    w = (torch.randint(-1, 2, (N, K), generator=gen) * (torch.rand(N, K, generator=gen) < 64.0 / K)).to(dtype)
    dy = torch.randint(-1, 2, (M, N), generator=gen) * (torch.rand(M, N, generator=gen) < min(1.0, 64.0 / N))
    dy = dy.to(dtype)

    def shifted(t):
        return torch.empty(t.numel() + 1, dtype=dtype, device="cuda")[1:].copy_(t.reshape(-1)).view(t.shape)
    xg, wg, dyg = shifted(x), w.cuda(), shifted(dy)
    assert xg.data_ptr() % 16 == 2
    want = x.double() @ w.double().T
    assert torch.equal(ops.linear(xg, wg).cpu().double(), want)
    dx, dw, db = ops.linear_backward(xg, wg, dyg)
    assert torch.equal(dx.cpu().double(), dy.double() @ w.double())
    assert torch.equal(dw.cpu().double(), dy.double().T @ x.double())
    assert torch.equal(db.cpu().double(), dy.double().sum(0))
    lib, dt = _lib.load(), _lib.DDL_DT_BF16 if dtype == torch.bfloat16 else _lib.DDL_DT_F16
    assert lib.ddl_gemm_in_place(dt, 0, K, 1, K, 1, M, N, K) == 1
    elems = lib.ddl_gemm_workspace_at(dt, 0, K, 1, K, 1, M, N, K)
    for n in {0, elems // 2, elems}:
        work = torch.full((n,), float("nan"), device="cuda") if n else None
        out = torch.full((M, N), 77.0, dtype=dtype, device="cuda")
        rc = lib.ddl_gemm_ws(xg.data_ptr(), K, 1, wg.data_ptr(), K, 1, None, out.data_ptr(), dt, N, M, N, K,
                             None if work is None else work.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "ddl_gemm_ws")
        assert torch.equal(out.cpu().double(), want)


@pytest.mark.parametrize("a_t,b_t", [(False, True), (True, True)])
def test_gemm_16_bit_random_within_tolerance_and_ragged_depth(ops, a_t, b_t):
    """Random operands, a reduction length that is no multiple of the k-tile
    (and, with both operands read down their columns, of nothing at all)."""
    from distdl_amd import _lib
    M, N, K = 328, 272, (1000 if not a_t else 1003)
    gen = torch.Generator().manual_seed(K)
    a = torch.randn(M, K, generator=gen).to(torch.bfloat16)
    b = (0.02 * torch.randn(N, K, generator=gen)).to(torch.bfloat16)
    ag, a_rs, a_ks = _gemm_operand(a, a_t, 0)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, 0)
    out = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    rc = _lib.load().ddl_gemm(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, None, out.data_ptr(), _lib.DDL_DT_BF16, N,
                              M, N, K, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ddl_gemm")
    _lin_check(bits16(out), a, b, None)


@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,pad", [(4060, 1000, 40, 0), (4096, 4352, 132, 4), (16384, 256, 36, 8), (4100, 1004, 288, 0)])
def test_gemm_f32_large_products_read_every_operand_layout(ops, a_t, b_t, M, N, K, pad):
    """Products of some thousand rows or columns (tiles of 64 x 64 and of 128 x 128),
    in every combination of operand layouts, with integer operands: every sum is
    exact in fp32, so the result must equal the fp64 product -- tiles that
    straddle M, N and K, pitched operands.  (Integers this small are one bf16
    part; test_gemm_f32_by_exact_bf16_parts has all three.)"""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M + 3 * N + K + 2 * a_t + b_t)
    a = torch.randint(-3, 4, (M, K), generator=gen).float()
    b = torch.randint(-3, 4, (N, K), generator=gen).float()
    bias = torch.randint(-5, 6, (N,), generator=gen).float()
    ag, a_rs, a_ks = _gemm_operand(a, a_t, pad)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, pad)
    ldy = N + 4
    out = torch.full((M, ldy), 77.0, device="cuda")
    rc = _lib.load().ddl_gemm_f32(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, bias.cuda().data_ptr(), out.data_ptr(), ldy,
                                  M, N, K, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ddl_gemm_f32")
    want = a.double() @ b.double().T + bias.double()
    got = out.cpu().double()
    assert torch.equal(got[:, :N], want)
    assert (got[:, N:] == 77.0).all()


@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,pad,splits", [
    # tiles of 64 x 64, 32 x 64 and 32 x 32; odd lengths and pitches; one k-tile, a straddling one, an odd number of rounds
    (4, 4, 1, 0, False), (5, 7, 9, 1, False), (33, 31, 33, 3, False), (64, 64, 64, 0, False), (130, 65, 96, 5, False),
    (1030, 517, 131, 0, False), (2050, 1027, 100, 2, False),
    # the reduction split over groups of wavefronts, and over workgroups, unequal shares
    (201, 263, 1033, 1, False), (201, 263, 2501, 1, True), (64, 100, 4095, 0, True),
    # enough work for the 128 x 128 tiles
    (4096, 4352, 1540, 4, False)])
def test_gemm_f32_products_of_every_size_and_pitch(ops, a_t, b_t, M, N, K, pad, splits):
    """Integer operands (every sum is exact in fp32) at the sizes where the fp32 tiles can go wrong, with and
    without the workspace that lets them split the reduction, on buffers that end where the operands end."""
    from distdl_amd import _lib
    gen = torch.Generator().manual_seed(M + 3 * N + K + 2 * a_t + b_t)
    a = torch.randint(-3, 4, (M, K), generator=gen).float()
    b = torch.randint(-3, 4, (N, K), generator=gen).float()
    bias = torch.randint(-5, 6, (N,), generator=gen).float()
    ag, a_rs, a_ks = _gemm_operand(a, a_t, pad)
    bg, b_rs, b_ks = _gemm_operand(b, b_t, pad)
    want = a.double() @ b.double().T + bias.double()
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    elems = lib.ddl_gemm_workspace(_lib.DDL_DT_F32, a_rs, a_ks, b_rs, b_ks, M, N, K)
    assert (elems > 0) == splits
    ldy = N + 4 + (M & 1)
    for n in {0, elems}:
        work = torch.full((n,), float("nan"), device="cuda") if n else None
        out = torch.full((M, ldy), 77.0, device="cuda")
        rc = lib.ddl_gemm_ws(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, bias.cuda().data_ptr(), out.data_ptr(), _lib.DDL_DT_F32,
                             ldy, M, N, K, None if work is None else work.data_ptr(), n, stream)
        _lib.check(rc, "ddl_gemm_ws")
        got = out.cpu().double()
        assert torch.equal(got[:, :N], want)
        assert (got[:, N:] == 77.0).all()


class _Plan32(ctypes.Structure):
    _fields_ = [("groups", ctypes.c_int), ("edge", ctypes.c_int), ("us", ctypes.c_double), ("splits", ctypes.c_int), ("workspace", ctypes.c_int64)]


def _plan32(M, N, K, a_t=False, b_t=False):
    """What the library's dispatch (ddl::plan32) takes for an fp32 product of operands end to end on this GPU: `edge` 128 for
    the tiles of bf16 parts, else `groups` for the small ones."""
    from distdl_amd import _lib
    plan = _lib.load()._ZN3ddl6plan32Elllllllil
    plan.restype, plan.argtypes = _Plan32, [ctypes.c_int64] * 7 + [ctypes.c_int, ctypes.c_int64]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return plan(*((1, M) if a_t else (K, 1)), *((1, N) if b_t else (K, 1)), M, N, K, cus, 2 ** 62)


@pytest.mark.parametrize("M,N,K,splits", [
    # small tiles
    (1300, 1411, 3, 0), (1281, 1408, 15, 0), (1280, 1409, 16, 0), (1300, 1411, 17, 0), (1279, 1410, 33, 0), (1300, 1411, 79, 0), (129, 1411, 4099, 0),
    (2049, 130, 1000, 0), (128, 128, 8200, 0),
    # 128 x 128 tiles of bf16 parts
    (3300, 3411, 3, 1), (3281, 3408, 15, 1), (3280, 3409, 16, 1), (3300, 3411, 17, 1), (3279, 3410, 33, 1), (3300, 3411, 79, 1), (3300, 3411, 100, 1),
    (257, 3411, 4099, 3), (2049, 513, 2000, 3), (640, 640, 8200, 8)])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
def test_gemm_f32_by_exact_bf16_parts(ops, a_t, b_t, M, N, K, splits):
    """Products large enough for 128 x 128 tiles on the bf16 matrix cores: partial tiles, every remainder of the k-tiles, the
    reduction in one piece and split, rows of odd length that start anywhere, operands as they lie; and products next to them
    that small tiles take.  The error against float64 is that of fp32 sums, and no larger than the fp32 matrix instruction's
    was (1.5e-6 for the longest of these sums, in the 2-norm)."""
    plan = _plan32(M, N, K, a_t, b_t)
    assert (plan.edge, plan.splits if plan.edge else 0) == ((128, splits) if splits else (0, 0))
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)

    def operand(rows, transposed):
        shape = (K, rows) if transposed else (rows, K)
        store = torch.full((shape[0] * (shape[1] + 3) + 1,), float("nan"), device="cuda")
        t = store[1:].as_strided(shape, (shape[1] + 3, 1), 1)
        t.copy_(torch.randn(shape, generator=gen, device="cuda"))
        return t, (1, shape[1] + 3) if transposed else (shape[1] + 3, 1)
    a, sa = operand(M, a_t)
    b, sb = operand(N, b_t)
    bias = torch.randn(N, generator=gen, device="cuda")
    out = torch.empty(M, N, device="cuda")
    ops._gemm(a, *sa, b, *sb, bias, out, ops._LINEAR_DTYPES[torch.float32], M, N, K)
    a64, b64 = (a.t() if a_t else a).double(), (b.t() if b_t else b).double()
    want = a64 @ b64.t() + bias.double()
    assert float((out.double() - want).norm() / want.norm()) <= 1.5e-6
    assert bool(((out.double() - want).abs() <= (K + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs().t() + bias.double().abs())).all())


@pytest.mark.parametrize("M,N,K,edge", [(1400, 1400, 48, 0), (1400, 1400, 1000, 0), (3300, 3300, 48, 128), (3300, 3300, 1000, 128)])
def test_gemm_f32_of_values_that_bf16_parts_cannot_carry(ops, M, N, K, edge):
    """Infinities, NaN, values next to the largest float and large ones, rows so small that their parts would be denormal, and zeros: the
    products are those of fp32 arithmetic, and tiles without such values are not touched by the others."""
    assert _plan32(M, N, K).edge == edge
    gen = torch.Generator(device="cuda").manual_seed(K)
    x, w = torch.randn(M, K, generator=gen, device="cuda"), torch.randn(N, K, generator=gen, device="cuda")
    plain = ops.linear(x, w)
    x[5, 3], x[6, 4], x[140, 7] = float("inf"), float("-inf"), float("nan")
    x[300] *= 2.0 ** -120
    x[301] = 0
    x[600] = 2.0 ** 127 * 1.99999
    w[0] = 1.0                    # exactly bf16: its smaller parts are zero, and infinity times zero is not a number
    w[1] = 0
    w[900] *= 2.0 ** -110
    w[1399, 0] = 1e37
    got = ops.linear(x, w).cpu()
    want = x.cpu().double() @ w.cpu().double().t()
    as32 = want.float()           # overflow to infinity as fp32 has it, where no partial sum is close to it
    size = x.cpu().double().abs() @ w.cpu().double().abs().t()
    sure = ~((size > 3.0e38) & (size < float("inf")))
    assert torch.equal(got.isnan()[sure], as32.isnan()[sure]) and torch.equal(got.isinf()[sure], as32.isinf()[sure])
    assert torch.equal(got[as32.isinf() & sure], as32[as32.isinf() & sure])
    ok = sure & as32.isfinite()
    assert bool(((got.double() - want).abs()[ok] <= (K + 2) * 2.0 ** -24 * size[ok] + 2.0 ** -149 * K).all())
    untouched = torch.ones(M, dtype=torch.bool)
    untouched[:256] = untouched[256:384] = untouched[512:640] = False     # the tiles' rows
    columns = torch.ones(N, dtype=torch.bool)
    columns[:128] = columns[896:1024] = columns[1280:1408] = False
    assert torch.equal(got[untouched][:, columns], plain.cpu()[untouched][:, columns])


def _sums_of_fp32(x, w):
    """x w^T with one rounding to fp32 per term, in the order of k."""
    out = torch.zeros(x.shape[0], w.shape[0], device="cuda")
    for k in range(x.shape[1]):
        out = (out.double() + x[:, k, None].double() * w[None, :, k].double()).float()
    return out


@pytest.mark.parametrize("density", [1.0, 0.25, 0.1, 0.01, 0])
@pytest.mark.parametrize("M,N,K,a_t,b_t,edge", [(3300, 3411, 100, False, False, 128), (3300, 3411, 100, True, True, 128), (640, 640, 8200, False, True, 128)])
def test_gemm_f32_error_of_sparse_operands(ops, M, N, K, a_t, b_t, edge, density):
    """Sums of few terms that are not zero: adding zeros rounds nothing in fp32 arithmetic, so the error against float64 is to
    stay below that of one rounding to fp32 per term.  With one such term in a row (density 0) the result is its product,
    rounded once; on bf16 parts the sum of the smaller parts is rounded eight times besides, at less than 2^-7 of the result,
    which moves that rounding by 2^-4 of its unit at most."""
    assert _plan32(M, N, K, a_t, b_t).edge == edge
    gen = torch.Generator(device="cuda").manual_seed(K)
    x, w = torch.randn(M, K, generator=gen, device="cuda"), torch.randn(N, K, generator=gen, device="cuda")
    if density == 0:
        x *= torch.nn.functional.one_hot(torch.randint(0, K, (M,), generator=gen, device="cuda"), K)
    else:
        x *= torch.rand(M, K, generator=gen, device="cuda") < density
    a, sa = (x.t().contiguous(), (1, M)) if a_t else (x, (K, 1))
    b, sb = (w.t().contiguous(), (1, N)) if b_t else (w, (K, 1))
    out = torch.empty(M, N, device="cuda")
    ops._gemm(a, *sa, b, *sb, None, out, ops._LINEAR_DTYPES[torch.float32], M, N, K)
    want = x.double() @ w.double().t()
    error = out.double() - want
    if density == 0:
        assert bool((error.abs() <= (1 + 2.0 ** -4) * 2.0 ** -24 * want.abs()).all())
    else:
        assert float(error.norm()) <= float((_sums_of_fp32(x, w).double() - want).norm())


@pytest.mark.parametrize("M,N,K,a_t,b_t,edge", [(3300, 3411, 48, False, False, 128), (3300, 3411, 100, True, True, 128), (640, 640, 8200, False, True, 128),
                                                (1300, 1411, 48, False, False, 0)])
def test_gemm_f32_of_rows_of_mixed_magnitudes(ops, M, N, K, a_t, b_t, edge):
    """Elements of one row from the smallest denormal to ordinary ones, next to zeros: every product is as exact as in fp32
    arithmetic, also where the small elements alone meet large ones of the other operand and make up the result."""
    assert _plan32(M, N, K, a_t, b_t).edge == edge
    gen = torch.Generator(device="cuda").manual_seed(K)

    def mixed(rows, least, most):
        exponent = torch.randint(least, most + 1, (rows, K), generator=gen, device="cuda")
        keep = torch.rand(rows, K, generator=gen, device="cuda") < 0.1
        return (torch.randn(rows, K, generator=gen, device="cuda", dtype=torch.float64) * torch.pow(2.0, exponent.double()) * keep).float()
    x, w = mixed(M, -149, 4), mixed(N, -20, 60)
    x[:128, 0], w[:, 0] = 1.0, 0.0
    x[:128, 1:] = 0.0
    x[:128, 1] = torch.randn(128, generator=gen, device="cuda") * 2.0 ** -118        # the whole result of these rows ...
    w[:64, 1] = torch.randn(64, generator=gen, device="cuda") * 2.0 ** 97            # ... with parts of bf16
    w[256:300, 1] = torch.randn(44, generator=gen, device="cuda") * 2.0 ** 117       # ... and with elements too large for them
    a, sa = (x.t().contiguous(), (1, M)) if a_t else (x, (K, 1))
    b, sb = (w.t().contiguous(), (1, N)) if b_t else (w, (K, 1))
    out = torch.empty(M, N, device="cuda")
    ops._gemm(a, *sa, b, *sb, None, out, ops._LINEAR_DTYPES[torch.float32], M, N, K)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((out.double() - want).abs() <= (K + 2) * 2.0 ** -24 * size + 2.0 ** -149 * K).all())
    one = (x[:128] != 0).sum(1) == 2                 # 1 and the small element: one product
    narrow = (out.double() - want).abs()[:128][one][:, :300]
    assert bool((narrow <= (1 + 2.0 ** -4) * 2.0 ** -24 * size[:128][one][:, :300] + 2.0 ** -149).all())


def test_gemm_f32_large_products_random_and_odd_depth(ops):
    """Random operands through the 128 x 128 tiles: both operands read along
    their rows, so the reduction length may be anything (here 1003, no multiple
    of the k-tile or of a vector); and the forward layout with K = 1000."""
    from distdl_amd import _lib
    for a_t, b_t, K in ((True, True, 1003), (False, False, 1000)):
        M, N = 4096, 1024
        assert _plan32(M, N, K, a_t, b_t).edge == 128
        gen = torch.Generator().manual_seed(K)
        a = torch.randn(M, K, generator=gen)
        b = 0.02 * torch.randn(N, K, generator=gen)
        ag, a_rs, a_ks = _gemm_operand(a, a_t, 0)
        bg, b_rs, b_ks = _gemm_operand(b, b_t, 0)
        out = torch.empty((M, N), device="cuda")
        rc = _lib.load().ddl_gemm_f32(ag.data_ptr(), a_rs, a_ks, bg.data_ptr(), b_rs, b_ks, None, out.data_ptr(), N, M, N, K,
                                      torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "ddl_gemm_f32")
        want = a.double() @ b.double().T
        err = (out.cpu().double() - want).abs()
        # fp32 products and sums of K terms: relative to the size of the terms, a few ulp times sqrt(K)
        assert float(err.max()) <= 1e-5 * float(a.abs().mean() * b.abs().mean()) * K


def test_gemm_16_bit_refuses_what_it_cannot_read_in_place(ops):
    from distdl_amd import _lib
    lib = _lib.load()
    a = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    y = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    bf16 = _lib.DDL_DT_BF16
    # an operand read down its columns whose row count is no multiple of 8
    assert lib.ddl_gemm(a.data_ptr(), 1, 64, a.data_ptr(), 64, 1, None, y.data_ptr(), bf16, 64, 60, 64, 64, stream) == -3
    # no unit stride
    assert lib.ddl_gemm(a.data_ptr(), 2, 64, a.data_ptr(), 64, 1, None, y.data_ptr(), bf16, 64, 16, 64, 16, stream) == -5
    # reduction length that an operand read along k cannot take
    assert lib.ddl_gemm(a.data_ptr(), 64, 1, a.data_ptr(), 1, 64, None, y.data_ptr(), bf16, 64, 64, 64, 60, stream) == -3
    # pitch below the row count
    assert lib.ddl_gemm(a.data_ptr(), 1, 8, a.data_ptr(), 64, 1, None, y.data_ptr(), bf16, 64, 64, 64, 8, stream) == -1
    assert b"rows" in lib.ddl_last_error()
    torch.cuda.synchronize()


def test_linear_layers_forward(ops):
    """DistributedLinear and DistributedLinearAllGather (solo rank 0 of 8,
    weights split on out_features) call the same kernel."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLinear
    from distdl_amd.nn import DistributedLinearAllGather
    world = SimWorld(8)
    Pw = world.partition(0)
    P_x = Pw.create_partition_inclusive([0]).create_cartesian_topology_partition([1, 1])
    P_y = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([1, 8])
    P_w = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([8, 1])
    torch.manual_seed(6)
    layer = DistributedLinear(P_x, P_y, P_w, 256, 1024).to(torch.bfloat16)
    assert tuple(layer.sublinear.weight.shape) == (128, 256) and layer.sublinear.bias is not None
    x = torch.randn(64, 256).to(torch.bfloat16)
    with torch.no_grad():
        y = layer(x.cuda())
    _lin_check(bits16(y), x, layer.sublinear.weight.detach().cpu(), layer.sublinear.bias.detach().cpu())

    P_y3 = Pw.create_partition_inclusive(list(range(8))).create_cartesian_topology_partition([1, 1, 8])
    ag = DistributedLinearAllGather(P_y3, 256, 1024, dtype=torch.bfloat16)
    assert tuple(ag.weight.shape) == (1, 128, 256) and tuple(ag.bias.shape) == (1, 128, 1)
    x3 = torch.randn(2, 32, 256).to(torch.bfloat16)
    with torch.no_grad():
        y3 = ag(x3.cuda())
    assert y3.shape == (2, 32, 128)
    _lin_check(bits16(y3), x3, ag.weight.detach().cpu().view(128, 256), ag.bias.detach().cpu().view(128))


@pytest.mark.parametrize("P,x_shape,c_out", [
    ([1, 1], [2, 2], 4), ([1, 4], [1, 12], 16), ([1, 1, 4], [1, 8, 12], 16), ([2, 1, 4], [2, 4, 12], 16),
    ([1, 1, 1, 4], [1, 2, 4, 12], 16), ([1, 2, 1, 2], [2, 2, 4, 12], 16), ([2, 1, 1, 2], [2, 2, 4, 12], 16),
    ([2, 2, 1, 2], [2, 2, 4, 12], 16), ([2, 1, 3], [4, 5, 26], 20),
])
@pytest.mark.parametrize("use_bias", [False, True])
def test_linear_all_gather_layer_reference_layouts(ops, P, x_shape, c_out, use_bias):
    """DistributedLinearAllGather over all workers (loopback) on the partitions
    and shapes of the reference's adjoint tests (tests/layers/test_linear_ag.py:13-108:
    two to four dimensions, data-parallel axes beside the feature axis) and on
    an uneven one: the input is gathered along the features, every worker
    applies its rows of the weight (stored on the first line of workers,
    broadcast to the others), the output stays partitioned along the features.
    Forward and all three gradients against torch.nn.functional.linear on the
    whole tensors (float32, the reference's default)."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLinearAllGather
    from oracle import repartition as o_rep
    n, M, c_in = int(np.prod(P)), P[-1], x_shape[-1]
    gen = torch.Generator().manual_seed(sum(P) * 10 + len(P) + use_bias)
    x = torch.randn(*x_shape, generator=gen)
    w = 0.2 * torch.randn(c_out, c_in, generator=gen)
    b = 0.2 * torch.randn(c_out, generator=gen) if use_bias else None
    dy = torch.randn(*x_shape[:-1], c_out, generator=gen)
    xs = o_rep.scatter(x.numpy(), P)
    dys = o_rep.scatter(dy.numpy(), P)
    w_rows = o_rep.scatter(w.numpy(), [M, 1])
    b_rows = o_rep.scatter(b.numpy(), [M]) if use_bias else None

    def body(P_world):
        P_y = P_world.create_partition_inclusive(list(range(n))).create_cartesian_topology_partition(P)
        layer = DistributedLinearAllGather(P_y, c_in, c_out, bias=use_bias)
        stores = layer.P_store_weight.active
        if stores:
            m = int(layer.P_store_weight.index[-2])
            assert m == int(P_y.index[-1]) and all(int(i) == 0 for i in P_y.index[:-1])
            with torch.no_grad():
                layer.weight.copy_(torch.from_numpy(w_rows[m]).view(layer.weight.shape))
                if use_bias:
                    layer.bias.copy_(torch.from_numpy(b_rows[m]).view(layer.bias.shape))
        xin = torch.from_numpy(xs[P_y.rank]).cuda().requires_grad_(True)
        y = layer(xin)
        y.backward(torch.from_numpy(dys[P_y.rank]).cuda())
        torch.cuda.synchronize()
        dw = layer.weight.grad.cpu() if stores else None
        db = layer.bias.grad.cpu() if stores and use_bias else None
        return y.detach().cpu(), xin.grad.cpu(), dw, db, int(P_y.index[-1])

    outs = SimWorld(n).run(body)
    xr = x.clone().requires_grad_(True)
    wr = w.clone().requires_grad_(True)
    br = b.clone().requires_grad_(True) if use_bias else None
    yr = F.linear(xr, wr, br)
    yr.backward(dy)
    want_y = o_rep.scatter(yr.detach().numpy(), P)
    want_dx = o_rep.scatter(xr.grad.numpy(), P)
    want_dw = o_rep.scatter(wr.grad.numpy(), [M, 1])
    want_db = o_rep.scatter(br.grad.numpy(), [M]) if use_bias else None
    seen = 0
    for r, (y, dx, dw, db, m) in enumerate(outs):
        assert np.allclose(y.numpy(), want_y[r], rtol=1e-5, atol=1e-5)
        assert np.allclose(dx.numpy(), want_dx[r], rtol=1e-5, atol=1e-5)
        if dw is not None:
            seen += 1
            assert np.allclose(dw.numpy().reshape(-1, c_in), want_dw[m], rtol=1e-5, atol=1e-4)
            if use_bias:
                assert np.allclose(db.numpy().reshape(-1), want_db[m], rtol=1e-5, atol=1e-4)
    assert seen == M


@pytest.mark.parametrize("P,x_shape,c_out", [
    ([1, 1], [2, 12], 16), ([1, 4], [1, 12], 16), ([1, 1, 4], [1, 8, 12], 16), ([2, 1, 4], [2, 4, 12], 16),
    ([1, 1, 1, 4], [1, 2, 4, 12], 16), ([1, 2, 1, 2], [2, 2, 4, 12], 16), ([2, 1, 1, 2], [2, 2, 4, 12], 16),
    ([2, 2, 1, 2], [2, 2, 4, 12], 16), ([2, 1, 2], [4, 5, 26], 21), ([1, 1, 3], [2, 5, 26], 21),
])
@pytest.mark.parametrize("use_bias", [False, True])
def test_linear_reduce_scatter_layer_matches_torch(ops, P, x_shape, c_out, use_bias):
    """DistributedLinearReduceScatter over all workers (loopback) on the
    partitions and shapes of the reference's adjoint tests
    (tests/layers/test_linear_rs.py:10-105) and on two whose feature counts do
    not divide evenly: every worker multiplies its slice of the input features
    by its weight shard, the partial products are summed and scattered along the
    output features.  Forward and backward against torch.nn.functional.linear on
    the whole tensors (float32, the reference's default; reference:
    nn/linear_rs.py:361-364)."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLinearReduceScatter
    from oracle import repartition as o_rep
    n, M, c_in = int(np.prod(P)), P[-1], x_shape[-1]
    gen = torch.Generator().manual_seed(sum(P) * 10 + len(P) + use_bias)
    x = torch.randn(*x_shape, generator=gen)
    w = 0.2 * torch.randn(c_out, c_in, generator=gen)
    b = 0.2 * torch.randn(c_out, generator=gen) if use_bias else None
    dy = torch.randn(*x_shape[:-1], c_out, generator=gen)
    xs = o_rep.scatter(x.numpy(), P)
    dys = o_rep.scatter(dy.numpy(), P)
    w_shards = o_rep.scatter(w.numpy(), [1, M])

    def body(P_world):
        P_x = P_world.create_partition_inclusive(list(range(n))).create_cartesian_topology_partition(P)
        layer = DistributedLinearReduceScatter(P_x, c_in, c_out, bias=use_bias)
        with torch.no_grad():
            if layer.P_weight.active:
                layer.weight.copy_(torch.from_numpy(w_shards[int(P_x.index[-1])]).view(layer.weight.shape))
            if use_bias and layer.P_store_bias.active:
                layer.bias.copy_(b.view(layer.bias.shape))
        xin = torch.from_numpy(xs[P_x.rank]).cuda().requires_grad_(True)
        y = layer(xin)
        y.backward(torch.from_numpy(dys[P_x.rank]).cuda())
        torch.cuda.synchronize()
        dw = layer.weight.grad.cpu() if layer.P_weight.active else None
        db = layer.bias.grad.cpu() if use_bias and layer.P_store_bias.active else None
        return y.detach().cpu(), xin.grad.cpu(), dw, db, int(P_x.index[-1])

    outs = SimWorld(n).run(body)
    xr = x.clone().requires_grad_(True)
    wr = w.clone().requires_grad_(True)
    br = b.clone().requires_grad_(True) if use_bias else None
    yr = F.linear(xr, wr, br)
    yr.backward(dy)
    want_y = o_rep.scatter(yr.detach().numpy(), P)
    want_dx = o_rep.scatter(xr.grad.numpy(), P)
    want_dw = o_rep.scatter(wr.grad.numpy(), [1, M])
    seen_w = 0
    for r, (y, dx, dw, db, col) in enumerate(outs):
        assert np.allclose(y.numpy(), want_y[r], rtol=1e-5, atol=1e-5)
        assert np.allclose(dx.numpy(), want_dx[r], rtol=1e-5, atol=1e-5)
        if dw is not None:
            seen_w += 1
            assert np.allclose(dw.numpy().reshape(c_out, -1), want_dw[col], rtol=1e-5, atol=1e-4)
        if db is not None:
            assert r == 0 and np.allclose(db.numpy().reshape(-1), br.grad.numpy(), rtol=1e-5, atol=1e-4)
    assert seen_w == M


def test_empty_inputs_give_empty_or_zero_outputs(ops):
    """No rows, no tokens: every entry point returns without a launch of size
    zero; gradients that are sums over nothing are zeros."""
    dev = "cuda"
    x = torch.empty(0, 256, device=dev)
    g, b = torch.ones(256, device=dev), torch.zeros(256, device=dev)
    assert ops.layer_norm(x, g, b, 1e-5).shape == (0, 256)
    stats = ops.ln_partial_stats(x)
    assert stats.shape == (0, 2)
    assert ops.ln_normalize_affine(x, stats.unsqueeze(0), [256], g, b, 1e-5).shape == (0, 256)
    mean = rstd = torch.empty(0, device=dev)
    dx, dg, db = ops.ln_backward_one_pass(x, x, mean, rstd, g, 1.0 / 256)
    assert dx.shape == (0, 256) and float(dg.abs().max()) == 0 and float(db.abs().max()) == 0
    table = torch.randn(16, 64, device=dev).to(torch.bfloat16)
    ids = torch.empty(0, dtype=torch.int64, device=dev)
    assert ops.embedding_gather(table, ids, 0, 16).shape == (0, 64)
    dw = ops.embedding_backward(torch.empty(0, 64, dtype=torch.bfloat16, device=dev), ids, 0, 16)
    assert dw.shape == (16, 64) and float(dw.float().abs().max()) == 0
    w = torch.randn(24, 64, device=dev).to(torch.bfloat16)
    bias = torch.randn(24, device=dev).to(torch.bfloat16)
    assert ops.linear(torch.empty(0, 64, dtype=torch.bfloat16, device=dev), w, bias).shape == (0, 24)
    dx, dw, db = ops.linear_backward(torch.empty(0, 64, dtype=torch.bfloat16, device=dev), w,
                                     torch.empty(0, 24, dtype=torch.bfloat16, device=dev))
    assert dx.shape == (0, 64) and float(dw.float().abs().max()) == 0 and float(db.float().abs().max()) == 0
