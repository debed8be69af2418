"""16-bit products of operands at any address and pitch: the tiles of 64 and of 128 rows and columns, whole and split reductions,
the k-tile that needs care, reductions shorter than a load.  (The small tiles' own cases are in test_gpu_layers.py.)"""

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
    return buf, buf.data_ptr() + 2 * shift, (1, ld) if transposed else (ld, 1)


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
