"""16-bit products of operands at any address and pitch: the tiles of 64 and of 128 rows and columns, whole and split reductions,
the k-tile that needs care, reductions shorter than a load; and the rings of the fp32 products.  (The small tiles' own cases are in
test_gpu_layers.py.)"""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _strided(t, transposed, pad, shift):
    """``t`` on the GPU with ``pad`` elements after each line, ``shift`` elements into its buffer and ending with it."""
    t = t.t().contiguous() if transposed else t
    ld = t.shape[1] + pad
    buf = torch.full((shift + (t.shape[0] - 1) * ld + t.shape[1],), float("nan"), dtype=t.dtype, device="cuda")
    view = buf[shift:].as_strided(t.shape, (ld, 1))
    view.copy_(t)
    return buf, buf.data_ptr() + t.element_size() * shift, (1, ld) if transposed else (ld, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,pad,shift", [
    # tiles of 128: one k-tile, whole ones, an odd number of them, K one before and after a k-tile; rows and columns one, seven
    # and 127 past a tile; reductions split over workgroups; then reductions of 1, 7 and 8
    (2049, 2055, 64, 0, 1), (2176, 2047, 63, 1, 0), (2055, 2049, 65, 0, 3), (3967, 1031, 192, 2, 1), (1001, 2051, 4001, 0, 0),
    (515, 777, 6839, 3, 5), (300, 4097, 1, 0, 1), (77, 130, 7, 1, 0), (130, 77, 8, 0, 1)])
def test_products_of_operands_at_any_address(dtype, a_t, b_t, M, N, K, pad, shift):
    """Integers, so every partial sum is exact (at most 2^8 in bfloat16): equal to the sums in 64 bits.  What surrounds the
    operands is NaN, the workspace too, and nothing outside the result is written."""
    from distdl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)

    def draw(rows, keep):
        t = torch.randint(-1, 2, (rows, K), generator=gen, device="cuda")
        return (t * (torch.rand(rows, K, generator=gen, device="cuda") < keep)).to(dtype)
    a, b, bias = draw(M, 1.0), draw(N, min(1.0, 48.0 / K)), torch.randint(-3, 4, (N,), generator=gen, device="cuda").to(dtype)
    want = a.double() @ b.double().T + bias.double()
    assert want.abs().max() <= 256
    buf_a, pa, (a_rs, a_ks) = _strided(a, a_t, pad, shift)
    buf_b, pb, (b_rs, b_ks) = _strided(b, b_t, pad, shift)
    lib, dt, ldy = _lib.load(), _lib.DDL_DT_BF16 if dtype == torch.bfloat16 else _lib.DDL_DT_F16, N + 3
    assert lib.ddl_gemm_in_place(dt, 0, a_rs, a_ks, b_rs, b_ks, M, N, K) == 1
    elems = lib.ddl_gemm_workspace_at(dt, 0, a_rs, a_ks, b_rs, b_ks, M, N, K)
    for n in {0, elems // 2, elems}:
        work = torch.full((n,), float("nan"), device="cuda") if n else None
        out = torch.full((M, ldy), 77.0, dtype=dtype, device="cuda")
        rc = lib.ddl_gemm_ws(pa, a_rs, a_ks, pb, b_rs, b_ks, bias.data_ptr(), out.data_ptr(), dt, ldy, M, N, K,
                             None if work is None else work.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "ddl_gemm_ws")
        assert torch.equal(out[:, :N].double(), want)
        assert (out[:, N:] == 77.0).all()


@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N", [(33, 31), (777, 333), (1024, 1021)])
def test_fp32_reductions_around_the_ring_of_stages(a_t, b_t, M, N):
    """Four, two and one group of wavefronts that take alternate k-tiles of 32 through rings of four: reductions that fill the
    rings or not, leave the last groups a tile less, end with a k-tile of one element or one short of a whole one.  Integers, so
    equal to the sums in 64 bits."""
    from distdl_amd import _lib
    lib = _lib.load()
    for tiles in (1, 3, 4, 5, 7, 9, 10, 16, 17, 19, 21, 34):
        for K in (32 * tiles - 1, 32 * tiles, 32 * tiles + 1):
            gen = torch.Generator(device="cuda").manual_seed(M + K)
            a, b = (torch.randint(-4, 5, (n, K), generator=gen, device="cuda").float() for n in (M, N))
            _, pa, (a_rs, a_ks) = kept_a = _strided(a, a_t, 0, 0)
            _, pb, (b_rs, b_ks) = kept_b = _strided(b, b_t, 1, 1)
            out = torch.full((M, N + 1), 77.0, device="cuda")
            rc = lib.ddl_gemm_ws(pa, a_rs, a_ks, pb, b_rs, b_ks, None, out.data_ptr(), _lib.DDL_DT_F32, N + 1, M, N, K, None, 0,
                                 torch.cuda.current_stream().cuda_stream)
            _lib.check(rc, "ddl_gemm_ws")
            assert torch.equal(out[:, :N].double(), a.double() @ b.double().T), K
            assert (out[:, N] == 77.0).all()
            del kept_a, kept_b


_ADJOINTS = [
    # one k-tile and one element more, 64 x 64 tiles, an odd length of every kind; 128 x 128 tiles of both products and of dx;
    # split reductions of either; many rows and few columns, without db in one launch; one row more than the column sums take
    # there; aligned throughout
    (8, 8, 8, 0, 0), (65, 64, 66, 1, 1), (97, 77, 603, 0, 0), (718, 821, 2056, 0, 3), (2048, 1024, 1024, 0, 0), (3001, 130, 257, 2, 0),
    (16384, 24, 40, 0, 0), (16385, 17, 33, 0, 1), (9, 5001, 1200, 0, 0), (1200, 9, 5001, 1, 0)]
_ADJOINTS_32 = [
    # too few rows and too many tiles for one launch, which go one after the other (the first two, the last); fewer elements than a
    # k-tile, split reductions, as many rows as the column sums take there and one more
    (2, 2, 2, 0, 0), (5, 3, 7, 1, 1), (33, 31, 35, 0, 0), (97, 77, 603, 0, 3), (777, 333, 1024, 0, 0), (104, 1256, 960, 0, 0), (108, 192, 5376, 2, 1),
    (2048, 24, 40, 0, 0), (2049, 17, 33, 0, 1), (512, 512, 512, 0, 0), (1500, 130, 257, 3, 0), (2500, 900, 300, 0, 0)]


# What one launch is made of, and the sizes that take it with room for all splits: (tiles of dx and dw, workgroups that share a
# reduction of each, db summed there too), see ddl_linear_backward_plan.
_PLANNED = [
    ((1, 1, 1, 1, 1), (65, 64, 66, 1, 1)), ((1, 1, 8, 1, 1), (8, 2064, 8, 3, 3)), ((1, 1, 1, 3, 1), (2412, 9, 9, 0, 1)),
    ((1, 1, 8, 2, 1), (512, 1928, 8, 3, 3)),        # dw's partial sums lie behind those of dx
    ((1, 2, 1, 1, 1), (8, 840, 6480, 1, 0)), ((1, 2, 1, 4, 1), (6324, 2436, 105, 0, 0)),
    ((2, 1, 1, 1, 1), (836, 8, 7779, 8, 8)), ((2, 1, 1, 3, 1), (16384, 310, 266, 8, 8)),   # as many rows as the column sums take there
    ((2, 2, 1, 1, 1), (472, 66, 7510, 3, 3)), ((2, 2, 1, 6, 1), (4098, 66, 1151, 0, 1)), ((2, 2, 2, 6, 1), (6844, 2509, 71, 0, 1)),
    ((1, 1, 1, 8, 0), (16385, 10, 8, 0, 0))]       # one row more
_PLANNED_32 = [
    ((1, 1, 1, 1, 1), (3, 8, 8, 1, 0)), ((1, 2, 1, 1, 1), (37, 8, 8, 1, 0)), ((1, 2, 1, 2, 1), (394, 8, 2105, 3, 3)),
    ((1, 2, 3, 1, 1), (1282, 1815, 199, 3, 3)), ((1, 4, 1, 1, 1), (67, 8, 9, 0, 1)), ((1, 4, 1, 8, 1), (2048, 16, 9, 0, 1)),
    ((2, 1, 1, 1, 1), (2, 33, 8, 3, 3)), ((2, 1, 2, 1, 1), (2, 232, 2852, 0, 0)), ((2, 2, 1, 1, 1), (38, 35, 9, 3, 3)),
    ((2, 2, 1, 2, 1), (255, 35, 1392, 1, 0)), ((2, 2, 2, 1, 1), (41, 232, 1406, 3, 3)), ((2, 2, 2, 2, 1), (267, 247, 508, 0, 0)),
    ((2, 4, 1, 1, 1), (78, 36, 10, 3, 3)), ((2, 4, 1, 6, 1), (1647, 36, 9, 0, 0)), ((2, 4, 8, 1, 1), (335, 1483, 34, 0, 0)),
    ((2, 4, 1, 8, 0), (2499, 33, 9, 8, 8)), ((4, 1, 1, 1, 1), (2, 81, 8, 0, 1)), ((4, 1, 4, 1, 1), (2, 1402, 10, 0, 1)),
    ((4, 2, 1, 1, 1), (34, 77, 9, 0, 1)), ((4, 2, 4, 1, 1), (36, 1322, 10, 1, 0)), ((4, 4, 1, 1, 1), (65, 77, 8, 3, 3)),
    ((4, 4, 1, 8, 1), (2028, 67, 8, 8, 8)), ((4, 4, 4, 1, 1), (71, 1411, 8, 0, 0)), ((4, 4, 6, 2, 1), (537, 1510, 11, 0, 1)),
    (None, (2500, 900, 300, 0, 0)), (None, (2, 2, 2, 0, 0))]


@pytest.mark.parametrize("dtype,plan,case", [(dt, *c) for dt in (torch.bfloat16, torch.float16) for c in _PLANNED] +
                         [(torch.float32, *c) for c in _PLANNED_32])
def test_every_form_of_the_adjoint_in_one_launch(dtype, plan, case):
    """The sizes go where this list says, and the results are exact there."""
    from distdl_amd import _lib
    M, N, K, pad, shift = case
    lib, dt = _lib.load(), {torch.bfloat16: _lib.DDL_DT_BF16, torch.float16: _lib.DDL_DT_F16, torch.float32: _lib.DDL_DT_F32}[dtype]
    sizes = (int(pad % 8 == 0 and shift % 8 == 0), M, N, K, K + pad, K + pad, N + pad)
    elems = lib.ddl_linear_backward_workspace_at(dt, *sizes, 1, 1, 1)
    got = (ctypes.c_int * 5)()
    taken = lib.ddl_linear_backward_plan(dt, *sizes, 1, elems, got)
    assert (tuple(got) if taken else None) == plan
    test_adjoint_of_a_linear_shard_in_one_launch(dtype, M, N, K, pad, shift)


@pytest.mark.parametrize("dtype,M,N,K,pad,shift", [(dt, *c) for dt in (torch.bfloat16, torch.float16) for c in _ADJOINTS] +
                         [(torch.float32, *c) for c in _ADJOINTS_32])
def test_adjoint_of_a_linear_shard_in_one_launch(dtype, M, N, K, pad, shift):
    """dx, dw and db on integers, equal to the sums in 64 bits; with the workspace asked for, half of it and none; what surrounds the
    operands is NaN, and the products alone, which take other kernels, give the same."""
    from distdl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)

    def draw(rows, cols, keep):
        t = torch.randint(-1, 2, (rows, cols), generator=gen, device="cuda")
        return (t * (torch.rand(rows, cols, generator=gen, device="cuda") < keep)).to(dtype)
    x, w, dy = draw(M, K, min(1.0, 40.0 / M)), draw(N, K, min(1.0, 40.0 / N)), draw(M, N, min(1.0, 2000.0 / M))
    want = [dy.double() @ w.double(), dy.double().T @ x.double(), dy.double().sum(0)]
    assert max(t.abs().max() for t in want) <= 256
    (bx, px, (ldx, _)), (bw, pw, (ldw, _)), (bd, pd, (ldd, _)) = [_strided(t, False, pad, shift) for t in (x, w, dy)]
    lib, dt = _lib.load(), {torch.bfloat16: _lib.DDL_DT_BF16, torch.float16: _lib.DDL_DT_F16, torch.float32: _lib.DDL_DT_F32}[dtype]
    aligned = int(pad == 0 and shift % 8 == 0)
    stream = torch.cuda.current_stream().cuda_stream
    for wanted in ((1, 1, 1), (1, 1, 0), (1, 0, 1), (0, 1, 0)):
        elems = lib.ddl_linear_backward_workspace_at(dt, aligned, M, N, K, ldx, ldw, ldd, *wanted)
        for n in {elems, elems // 2, 0} if wanted[2] == 0 or M <= 2048 else {elems}:
            work = torch.full((n,), float("nan"), device="cuda") if n else None
            outs = [torch.full((s + 8,), 77.0, dtype=dtype, device="cuda") if on else None for s, on in zip((M * K, N * K, N), wanted)]
            rc = lib.ddl_linear_backward(px, pw, pd, *[None if o is None else o.data_ptr() for o in outs], dt, M, N, K, ldx, ldw, ldd,
                                         None if work is None else work.data_ptr(), n, stream)
            _lib.check(rc, "ddl_linear_backward")
            for o, t in zip(outs, want):
                if o is not None:
                    assert torch.equal(o[:-8].view(t.shape).double(), t) and (o[-8:] == 77.0).all()
