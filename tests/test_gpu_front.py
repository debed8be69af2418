"""The native front ends against the general path behind them: the same bits for
every form that both take, and the same refusals."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]


class _Nothing:
    """An extension that answers None to everything but the boxes, which have no other path."""

    def __init__(self, real):
        self.Boxes = real.Boxes

    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture
def both(monkeypatch):
    """both(fn): fn() through the native front end and without it, the results equal bit for bit; returns them, or the type
    and message of the error that both raise.  ``taken`` counts the calls that the front end answered."""
    from distdl_amd import _lib
    real = _lib.front()

    class Counting:
        def __getattr__(self, name):
            f = getattr(real, name)

            def call(*args):
                res = f(*args)
                run.taken += res is not None
                return res
            return f if name == "Boxes" else call

    def outcome(fn, front):
        monkeypatch.setattr(_lib, "_front", front)
        try:
            res = fn()
        except Exception as e:
            return type(e), str(e)
        finally:
            monkeypatch.setattr(_lib, "_front", real)
        return res if isinstance(res, (list, tuple)) else [res]

    def run(fn):
        a, b = outcome(fn, Counting()), outcome(fn, _Nothing(real))
        assert len(a) == len(b)
        for p, q in zip(a, b):
            assert type(p) is type(q)
            if isinstance(p, torch.Tensor):
                assert p.shape == q.shape and p.dtype == q.dtype and p.stride() == q.stride()
                assert torch.equal(p.detach().contiguous().view(torch.uint8), q.detach().contiguous().view(torch.uint8))
            else:
                assert p == q
        return a
    run.taken = 0
    return run


def _randn(*shape, dtype=torch.float32, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed + sum(shape)), device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k,pitch", [((3,), 5, 7, 7), ((2, 9), 64, 128, 128), ((1,), 40, 72, 80), ((5, 1), 1, 33, 50), ((0,), 8, 16, 16),
                                         ((4,), 8, 0, 0), ((300,), 333, 1021, 1021), ((64,), 4096, 512, 512)])
def test_linear_and_its_adjoint(both, dtype, m, n, k, pitch):
    from distdl_amd import hip_ops
    w = _randn(n, pitch, dtype=dtype)[:, :k]
    b, x, dy = _randn(n, dtype=dtype), _randn(*m, k, dtype=dtype), _randn(*m, n, dtype=dtype, seed=1)
    both(lambda: hip_ops.linear(x, w, b))
    both(lambda: hip_ops.linear(x, w))
    for need in ((True, True, True), (True, False, False), (False, True, True), (False, False, True)):
        both(lambda: hip_ops.linear_backward(x, w, dy, *need))
    if x.numel() and (dtype == torch.float32 or all(v % 8 == 0 for v in (n, k, pitch))):
        assert both.taken == 6
    # operands that are not contiguous, off a 16-byte boundary, of other types or other lengths, on the host
    off = torch.empty(x.numel() + 1, dtype=dtype, device="cuda")[1:].view(x.shape).copy_(x)
    both(lambda: hip_ops.linear(off, w, b))
    both(lambda: hip_ops.linear_backward(off, w, dy))
    both(lambda: hip_ops.linear(x.transpose(0, -1).contiguous().transpose(0, -1), w, b))
    both(lambda: hip_ops.linear(x, w.t().contiguous().t(), b))
    both(lambda: hip_ops.linear_backward(x, w, dy.transpose(0, -1).contiguous().transpose(0, -1)))
    taken = both.taken
    for bad in (lambda: hip_ops.linear(x.double(), w), lambda: hip_ops.linear(x, w.double()), lambda: hip_ops.linear(x, w, b.double()),
                lambda: hip_ops.linear(x, w, b[:-1]), lambda: hip_ops.linear(x, w[0]), lambda: hip_ops.linear(x[..., :-1], w),
                lambda: hip_ops.linear(x.cpu(), w), lambda: hip_ops.linear(x, w.cpu()), lambda: hip_ops.linear_backward(x, w, dy.double()),
                lambda: hip_ops.linear_backward(x, w, dy.cpu())):
        both(bad)
    assert both.taken == taken


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 1), (3, 5, 64), (7, 512), (9, 514), (6, 768), (33, 1024), (4, 1028), (5, 2050), (3, 8192), (2, 8194), (2, 16384), (2, 16388), (0, 64)])
@pytest.mark.parametrize("affine", [True, False])
def test_layer_norm_layer_and_its_adjoint(both, dtype, shape, affine):
    """Whole rows, at the widths where the adjoint takes another kernel, with and without parameters, gradients wanted of some."""
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.nn import DistributedLayerNorm
    P = SimWorld(1).partition(0).create_partition_inclusive([0]).create_cartesian_topology_partition([1] * len(shape))
    layer = DistributedLayerNorm(P, [shape[-1]], elementwise_affine=affine, dtype=dtype)
    if affine:
        with torch.no_grad():
            layer.weight.copy_(1 + 0.1 * _randn(*layer.weight.shape, seed=2))
            layer.bias.copy_(0.1 * _randn(*layer.bias.shape, seed=3))
    x, dy = _randn(*shape, dtype=dtype).requires_grad_(True), _randn(*shape, dtype=dtype, seed=1)

    def step(x, dy, wanted):
        y = layer(x)
        return [y, *torch.autograd.grad(y, wanted, dy)]
    params = [layer.weight, layer.bias] if affine else []
    for wanted in ([x] + params, [x], params[:1]):
        if wanted:
            both(lambda: step(x, dy, wanted))
    turned = x.detach().transpose(0, 1).contiguous().transpose(0, 1).requires_grad_(True)
    both(lambda: step(turned, dy, [turned] + params))
    both(lambda: step(x, dy.transpose(0, 1).contiguous().transpose(0, 1), [x] + params))
    both(lambda: step(x, dy[:1].expand(shape) if shape[0] else dy, [x] + params))
    if x.numel() and affine:
        assert both.taken >= 4


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,cols", [(1, 3), (70, 256), (33, 683), (5, 1025)])
def test_layer_norm_adjoint_of_shared_rows(both, dtype, rows, cols):
    from distdl_amd import hip_ops
    dy, x, gamma = _randn(rows, cols, dtype=dtype), _randn(rows, cols, dtype=dtype, seed=1), _randn(cols, dtype=dtype)
    mean, rstd = _randn(rows), _randn(rows, seed=4).abs()
    parts = _randn(3, rows, 2)

    def step(dy, x, gamma, want_gamma=True, want_beta=True):
        sums, work = hip_ops.ln_backward_partial_params(dy, x, mean, rstd, gamma)
        return [sums, *hip_ops.ln_backward_input_params(dy, x, mean, rstd, gamma, parts, 0.25 / cols, work, want_gamma, want_beta)]
    both(lambda: step(dy, x, gamma))
    both(lambda: step(dy, x, None))
    both(lambda: step(dy, x, gamma, want_beta=False))
    assert both.taken == 6
    work = hip_ops.ln_backward_partial_params(dy, x, mean, rstd, gamma)[1]
    both(lambda: step(_randn(rows + 1, cols + 1, dtype=dtype)[:rows, :cols], x, gamma))
    both(lambda: step(dy, x.double(), gamma))
    both(lambda: step(dy, x, gamma.cpu()))
    # as many elements in another shape
    for other in dy.view(cols, rows), dy.view(1, rows, cols), dy.view(-1):
        for refused in (lambda: hip_ops.ln_backward_partial_params(other, x, mean, rstd, gamma),
                        lambda: hip_ops.ln_backward_input_params(other, x, mean, rstd, gamma, parts, 0.25 / cols, work)):
            assert both(refused)[0] is ValueError
    assert both.taken == 6 or rows == 1       # (one row is contiguous at any pitch)


@pytest.mark.parametrize("dtype", DTYPES + [torch.float64])
@pytest.mark.parametrize("idt", [torch.int64, torch.int32, torch.int16])
def test_embedding_and_its_adjoint(both, dtype, idt):
    from distdl_amd import hip_ops
    w, ids, dy = _randn(20, 12, dtype=dtype), torch.arange(30, device="cuda").reshape(5, 6).to(idt) % 27, _randn(5, 6, 12, dtype=dtype)
    for t in (w, _randn(20, 15, dtype=dtype)[:, :12], w.t().contiguous().t(), w[:19], w.cpu()):
        both(lambda: hip_ops.embedding_gather(t, ids, 3, 23))
    known = idt != torch.int16
    assert both.taken == known                # the first
    both(lambda: hip_ops.embedding_gather(w, ids.t(), 3, 23))
    assert both.taken == known
    both(lambda: hip_ops.embedding_gather(w, ids[:0], 3, 23))
    assert both.taken == 2 * known
    for pad in (None, 5):
        both(lambda: hip_ops.embedding_backward(dy, ids, 3, 23, pad))
        both(lambda: hip_ops.embedding_backward(dy, ids, 3, 23, pad, True))
    adjoints = 4 * (known and dtype != torch.float64)
    assert both.taken == 2 * known + adjoints
    both(lambda: hip_ops.embedding_backward(dy.transpose(0, 2).contiguous().transpose(0, 2), ids, 3, 23))
    both(lambda: hip_ops.embedding_backward(dy, ids.t().contiguous().t(), 3, 23))
    both(lambda: hip_ops.embedding_backward(dy, ids[:4], 3, 23))
    assert both.taken == 2 * known + adjoints
    both(lambda: hip_ops.embedding_backward(dy[:0], ids[:0], 3, 23))
    both(lambda: hip_ops.embedding_backward(dy[..., :0], ids, 3, 23))


@pytest.mark.parametrize("dtype", DTYPES + [torch.float64, torch.int32, torch.int64, torch.uint8])
@pytest.mark.parametrize("axis", [0, 1, -1, 3])
@pytest.mark.parametrize("divisor", [1, 2, 3])
def test_gather_and_reduce_scatter_slabs(both, dtype, axis, divisor):
    from distdl_amd.backends.stub_hip import SimWorld
    from distdl_amd.backends.stub_hip.functional import all_gather
    world = SimWorld(3)
    P = world.partition(0).create_partition_inclusive([0, 1, 2]).create_cartesian_topology_partition([1, 1, 3])
    local = (10 * _randn(4, 7, 6)).to(dtype)
    pieces = {"all": [(10 * _randn(4, 7, 6, seed=q)).to(dtype) for q in range(3)]}
    world.transport.set_gather_provider("tag", lambda P, t: list(pieces["all"]))
    both(lambda: all_gather.gather_slabs(P, local, axis, "tag"))
    assert both.taken == (axis != 3)
    both(lambda: all_gather.reduce_scatter_slabs(P, local, axis, "tag", divisor))
    assert both.taken == 0 if axis == 3 else 2 - (dtype == torch.uint8)
    both(lambda: all_gather.gather_slabs(P, local.transpose(0, 2).contiguous().transpose(0, 2), axis, "tag"))
    both(lambda: all_gather.reduce_scatter_slabs(P, local.transpose(0, 2).contiguous().transpose(0, 2), axis, "tag", divisor))
    if axis == 1:       # pieces of different lengths, without elements, of another shape, off a 16-byte boundary of each other
        for odd in (pieces["all"][1][:, :3].contiguous(), pieces["all"][1][:, :0], pieces["all"][1][:3], pieces["all"][1].double(),
                    torch.empty(169, dtype=dtype, device="cuda")[1:].view(4, 7, 6).copy_(pieces["all"][1])):
            pieces["all"][1] = odd
            both(lambda: all_gather.gather_slabs(P, local, axis, "tag"))
            both(lambda: all_gather.reduce_scatter_slabs(P, local, axis, "tag", divisor))
