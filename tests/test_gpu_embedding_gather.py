"""The embedding's gather: rows of any length, address and element size, misses, more lanes than one launch numbers."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("idt", [torch.int64, torch.int32])
@pytest.mark.parametrize("n,dim,pad,shift", [
    # shorter than a vector, one vector and one element more or less, rows that end inside one, whole ones; workgroups of one row,
    # of many, with a part of a row; tables with a pitch and off a 16-byte boundary
    (1, 1, 0, 0), (1000, 3, 2, 1), (77, 7, 0, 0), (77, 8, 0, 0), (300, 9, 0, 3), (300, 15, 1, 0), (300, 16, 0, 0), (513, 17, 0, 1), (64, 64, 0, 0),
    (1000, 257, 3, 0), (9, 4095, 0, 0), (9, 4096, 0, 0), (3, 5000, 8, 1)])
def test_rows_of_any_length_and_address(dtype, idt, n, dim, pad, shift):
    from distdl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + dim)
    rows, lo, ld = 23, 5, dim + pad
    buf = torch.randint(0, 200, (shift + (rows - 1) * ld + dim,), generator=gen, device="cuda").to(dtype)
    table = buf[shift:].as_strided((rows, dim), (ld, 1))
    ids = torch.randint(0, 40, (n,), generator=gen, device="cuda").to(idt)
    hit = (ids >= lo) & (ids < lo + rows)
    want = torch.where(hit[:, None], table[(ids.long() - lo).clamp(0, rows - 1)], torch.zeros((), dtype=dtype, device="cuda"))
    for at in (0, 1):
        out = torch.full((at + n * dim + 8,), 77, dtype=dtype, device="cuda")
        rc = _lib.load().ddl_embedding_gather(table.data_ptr(), dim, ld, dtype.itemsize, ids.data_ptr(), int(idt == torch.int64), n, lo, lo + rows,
                                              out.data_ptr() + at * dtype.itemsize, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "ddl_embedding_gather")
        assert torch.equal(out[at:-8].view(n, dim), want) and (out[:at] == 77).all() and (out[-8:] == 77).all()


def test_more_lanes_than_one_launch_numbers():
    from distdl_amd import _lib
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB")
    n = (1 << 31) + 5
    table = torch.arange(256, device="cuda").to(torch.uint8)
    ids = torch.empty(n, dtype=torch.int32, device="cuda")
    for first in range(0, n, 1 << 29):
        part = ids[first:first + (1 << 29)]
        part.copy_(torch.arange(first, first + part.numel(), device="cuda") % 251)
    out = torch.full((n + 8,), 255, dtype=torch.uint8, device="cuda")
    rc = _lib.load().ddl_embedding_gather(table.data_ptr(), 1, 1, 1, ids.data_ptr(), 0, n, 0, 256, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ddl_embedding_gather")
    for first in range(0, n, 1 << 29):
        part = ids[first:first + (1 << 29)]
        assert torch.equal(out[first:first + part.numel()], part.to(torch.uint8))
    assert (out[n:] == 255).all()
