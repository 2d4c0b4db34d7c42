"""Dense -> CSR at the sizes where its row segments (2048 elements, one wavefront each, batches of 512)
begin and end, against numpy, bit for bit, through both entry points (needs an MI355X)."""
import ctypes as C

import numpy as np
import pytest

import fastdose_amd as fd
from fastdose_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def convert(torch, name, d, nnz):
    rows, cols = d.shape
    off = torch.full((rows + 1,), -7, dtype=torch.int64, device="cuda")
    col = torch.full((nnz + 1,), -1, dtype=torch.int64, device="cuda")
    val = torch.full((nnz + 1,), -1.0, dtype=torch.float32, device="cuda")
    csr = _lib.CSR(0, 0, nnz, off.data_ptr(), col.data_ptr(), val.data_ptr())
    _lib.call(name, C.c_void_p(d.data_ptr()), rows, cols, C.byref(csr), None)
    assert csr.nnz == nnz and int(col[nnz]) == -1 and float(val[nnz]) == -1.0
    return off, col[:nnz], val[:nnz]


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 2047), (1, 2048), (1, 2049), (3, 511), (3, 513), (5, 4096),
                                       (7, 4097), (257, 63), (2, 100_003), (1025, 2050)])
def test_segments(torch_cuda, rows, cols):
    torch = torch_cuda
    rng = np.random.default_rng([rows, cols])
    m = np.where(rng.random((rows, cols)) < 0.3, rng.standard_normal((rows, cols)), 0.0).astype(np.float32)
    m[0, 0], m[-1, -1] = 1.5, np.nan          # NaN counts as a nonzero, -0 as a zero
    if cols > 2:
        m[0, 1], m[-1, 1] = -0.0, -np.inf
    keep = m != 0
    r, c = np.nonzero(keep)
    for name in ("fd_dense_to_csr", "fd_dense_to_csr_noalloc"):
        off, col, val = convert(torch, name, torch.from_numpy(m).cuda(), len(c))
        assert np.array_equal(off.cpu().numpy(), np.concatenate([[0], np.cumsum(keep.sum(1))]))
        assert np.array_equal(col.cpu().numpy(), c)
        assert np.array_equal(val.cpu().numpy().view(np.uint32), m[r, c].view(np.uint32))


def test_more_segments_than_the_fixed_scratch_holds(torch_cuda):
    """2^20 rows of two segments each: the allocation-free entry point takes longer segments instead."""
    torch = torch_cuda
    rows, cols = 1 << 20, 2049
    d = torch.zeros((rows, cols), device="cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    at = torch.randperm(rows, generator=g, device="cuda")[:5000]
    where = torch.cat([at * cols + torch.randint(cols, (5000,), generator=g, device="cuda"),
                       at[:100] * cols + cols - 1]).unique()  # sorted
    d.view(-1)[where] = 2.0
    row = where // cols
    counts = torch.bincount(row, minlength=rows)
    off_want = torch.cat([counts.new_zeros(1), counts.cumsum(0)])
    for name in ("fd_dense_to_csr", "fd_dense_to_csr_noalloc"):
        off, col, val = convert(torch, name, d, len(where))
        assert torch.equal(off, off_want) and torch.equal(col, where % cols) and bool((val == 2.0).all())
