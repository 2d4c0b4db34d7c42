"""The voxel-major operator (fd_spmm_create) and its product over the shapes at which its kernels
branch (needs an MI355X): column tiles of 2048, row blocks of 64, rows with more than 64 entries in a
tile, rows in unsorted order and rows too short for the tile table (the general path), and every
arrangement of the product's lanes, against numpy in FP64."""
import ctypes as C

import numpy as np
import pytest

import fastdose_amd as fd
from fastdose_amd import _lib

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # unit roundoff of FP32


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def random_rows(rng, R, cols, fill, long_row=False):
    """(offsets, columns, values) of R rows with ascending columns: a run per row, a scatter of others,
    empty rows among them; long_row: row R // 2 holds every column."""
    offs, cs, vs = [0], [], []
    for r in range(R):
        n = int(rng.integers(0, max(2, int(2 * fill * cols))))
        start = int(rng.integers(0, cols))
        c = np.unique(np.concatenate([rng.integers(0, cols, n), np.arange(start, min(cols, start + n))]))
        if r % 7 == 3:
            c = c[:0]
        if long_row and r == R // 2:
            c = np.arange(cols)
        cs.append(c)
        vs.append(rng.uniform(0.01, 1.0, len(c)).astype(np.float32))
        offs.append(offs[-1] + len(c))
    return np.array(offs), np.concatenate(cs).astype(np.int64), np.concatenate(vs)


def dose_mat(torch, cols, mats):
    dm = fd.DoseMat(cols)
    for off, c, v in mats:
        d = [torch.as_tensor(np.ascontiguousarray(a)).cuda() for a in (off.astype(np.int64), c, v)]
        csr = fd.CSR(len(off) - 1, len(c), len(c), *(t.data_ptr() for t in d))
        torch.cuda.synchronize()
        _lib.call("fd_dosemat_add_csr", dm._h, C.byref(csr), None)
    return dm


def dense(mats, cols):
    out = []
    for off, c, v in mats:
        m = np.zeros((len(off) - 1, cols), np.float64)
        for r in range(len(off) - 1):
            m[r, c[off[r]:off[r + 1]]] = v[off[r]:off[r + 1]]
        out.append(m)
    return np.concatenate(out, 0)


def rounded(D, vtype):
    """The values the operator stores: FP32, or 16 bits of value / row maximum times the FP32 maximum."""
    if vtype == fd.FD_VAL_F32:
        return D
    s = D.max(1, keepdims=True).astype(np.float32)
    t = np.divide(D.astype(np.float32), s, out=np.zeros(D.shape, np.float32), where=s > 0)
    if vtype == fd.FD_VAL_FP16:
        q = t.astype(np.float16).astype(np.float32)
    else:
        u = t.view(np.uint32).astype(np.uint64)
        q = (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)
    return (q * s).astype(np.float64)


@pytest.mark.parametrize("vtype", [fd.FD_VAL_F32, fd.FD_VAL_BF16, fd.FD_VAL_FP16])
@pytest.mark.parametrize("R,cols,fill", [(1, 1, 1.0), (1, 2047, 0.3), (63, 2048, 0.02), (64, 2049, 0.1),
                                         (65, 4097, 0.05), (130, 6145, 0.02), (200, 40000, 0.004)])
def test_operator_holds_every_entry_in_row_order(torch_cuda, vtype, R, cols, fill):
    """D^T times the identity is D^T itself, each entry exactly (one term per sum)."""
    torch = torch_cuda
    rng = np.random.default_rng([R, cols, vtype])
    mats = [random_rows(rng, R, cols, fill, long_row=True), random_rows(rng, 3, cols, fill)]
    D = rounded(dense(mats, cols), vtype)
    dm = dose_mat(torch, cols, mats)
    with fd.Spmm(dm, vtype) as op:
        y = op.run(torch.eye(R + 3, device="cuda")).cpu().numpy()
    assert np.array_equal(y.T.astype(np.float64), D)


def test_general_path_gives_the_same_operator(torch_cuda):
    """Rows with their entries in another order, and rows of two entries in a wide volume, take the
    general path; its product equals the tiles' bit for bit where both can be built."""
    torch = torch_cuda
    rng = np.random.default_rng(5)
    off, c, v = random_rows(rng, 70, 5000, 0.03)
    order = np.concatenate([off[r] + rng.permutation(off[r + 1] - off[r]) for r in range(70)])
    x = torch.rand((70, 9), device="cuda")
    y = []
    for m in ((off, c, v), (off, c[order], v[order])):
        with fd.Spmm(dose_mat(torch, 5000, [m])) as op:
            y.append(op.run(x).cpu().numpy())
    assert np.array_equal(*y)
    cols, R = 3_000_000, 400
    c = np.sort(rng.choice(cols, (R, 2)), 1).astype(np.int64)
    c[:, 1] += c[:, 1] == c[:, 0]
    c = np.minimum(c, cols - 1)
    v = rng.uniform(0.01, 1.0, 2 * R).astype(np.float32)
    with fd.Spmm(dose_mat(torch, cols, [(np.arange(0, 2 * R + 1, 2), c.reshape(-1), v)])) as op:
        x = torch.rand((R, 1), device="cuda")
        got = op.run(x).cpu().numpy()[:, 0].astype(np.float64)
    want = np.zeros(cols)
    np.add.at(want, c.reshape(-1), v.astype(np.float64) * np.repeat(x.cpu().numpy()[:, 0].astype(np.float64), 2))
    assert np.all(np.abs(got - want) <= 4 * U * want)


@pytest.mark.parametrize("cols", [16383, 16384, 16385, 40961, 4096 ** 2, 4096 ** 2 + 1])
def test_scan_of_column_counts(torch_cuda, cols):
    """The general path scans one count per column: by one workgroup, in two kernels, in three."""
    torch = torch_cuda
    rng = np.random.default_rng(cols)
    R = 300
    c = np.sort(rng.choice(cols, (R, 2)), 1).astype(np.int64)
    c[0] = [0, cols - 1]
    c[:, 0] = np.where(c[:, 0] == c[:, 1], (c[:, 0] + 1) % cols, c[:, 0])
    c = c[:, ::-1].copy()  # not ascending
    v = rng.uniform(0.01, 1.0, 2 * R).astype(np.float32)
    with fd.Spmm(dose_mat(torch, cols, [(np.arange(0, 2 * R + 1, 2), c.reshape(-1), v)])) as op:
        x = torch.rand((R, 1), device="cuda")
        got = op.run(x).cpu().numpy()[:, 0].astype(np.float64)
    want = np.zeros(cols)
    np.add.at(want, c.reshape(-1), v.astype(np.float64) * np.repeat(x.cpu().numpy()[:, 0].astype(np.float64), 2))
    assert np.all(np.abs(got - want) <= 2 * R * U * want)


@pytest.mark.parametrize("R,cols", [(1472, 2048), (1473, 2049), (1985, 4096), (4100, 40 * 2048 + 1)])
def test_rows_beyond_one_list(torch_cuda, R, cols):
    """Up to 1984 rows that reach a tile are listed at once, 512 rows of the matrix at a time: all rows
    reach the first tile here, most with a few entries and some with all its columns (32 units of 64).
    The general path, which takes them in another order, is the reference: same bits."""
    torch = torch_cuda
    rng = np.random.default_rng([R, cols])
    rows = []
    for r in range(R):
        c = np.concatenate([rng.integers(0, 2048, 4), rng.integers(0, cols, 3)])
        if r % 200 == 77:
            c = np.arange(min(cols, 2048))
        rows.append(np.unique(c))
    off = np.concatenate([[0], np.cumsum([len(c) for c in rows])])
    c = np.concatenate(rows).astype(np.int64)
    v = rng.uniform(0.01, 1.0, len(c)).astype(np.float32)
    back = np.concatenate([np.arange(off[r], off[r + 1])[::-1] for r in range(R)])
    x = torch.rand((R, 3), device="cuda")
    y = []
    for m in ((off, c, v), (off, c[back], v[back])):
        with fd.Spmm(dose_mat(torch, cols, [m])) as op:
            y.append(op.run(x).cpu().numpy())
    assert np.array_equal(*y)
    D = np.zeros(cols)
    np.add.at(D, c, v.astype(np.float64) * np.repeat(x[:, 0].cpu().numpy().astype(np.float64), np.diff(off)))
    assert np.allclose(y[0][:, 0], D, rtol=R * U)


@pytest.mark.parametrize("R,cols", [(1, 1), (255, 257), (4096, 1025), (4097, 1025)])
def test_one_vector_and_16_bit_values(torch_cuda, R, cols):
    """Up to 4096 rows the products of scales and vector lie in LDS, shared by 1024 columns."""
    torch = torch_cuda
    rng = np.random.default_rng([R, cols])
    mats = [random_rows(rng, R, cols, 4.0 / cols, long_row=True)]
    x = rng.uniform(-1.0, 1.0, (R, 1)).astype(np.float32)
    dm = dose_mat(torch, cols, mats)
    for vtype in (fd.FD_VAL_BF16, fd.FD_VAL_FP16):
        D = rounded(dense(mats, cols), vtype)
        with fd.Spmm(dm, vtype) as op:
            y = op.run(torch.as_tensor(x).cuda()).cpu().numpy()
        want, mag = D.T @ x.astype(np.float64), np.abs(D).T @ np.abs(x.astype(np.float64))
        n = (D != 0).sum(0)[:, None]
        assert np.all(np.abs(y - want) <= (n + 3) * U * mag), vtype


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 8, 12, 16, 20, 31, 33, 64, 65, 100, 128, 130, 132, 256, 260])
def test_product_over_lane_arrangements(torch_cuda, k):
    """Sparse, medium and crowded stretches of columns (each picks its own lanes per column, the crowded
    one is split over the workgroup), a last partial tile, all value types."""
    torch = torch_cuda
    rng = np.random.default_rng(k)
    R, cols = 300, 1000
    p = np.concatenate([np.full(256, 0.003), np.full(300, 0.03), np.full(200, 0.12), np.full(244, 0.7)])
    M = np.where(rng.random((R, cols)) < p, rng.uniform(0.01, 1.0, (R, cols)), 0.0).astype(np.float32)
    M[:, 64:128] = 0.0
    r, c = np.nonzero(M)
    off = np.concatenate([[0], np.cumsum((M != 0).sum(1))])
    dm = dose_mat(torch, cols, [(off, c.astype(np.int64), M[r, c])])
    x = rng.uniform(-1.0, 1.0, (R, k)).astype(np.float32)
    for vtype in (fd.FD_VAL_F32, fd.FD_VAL_BF16, fd.FD_VAL_FP16):
        D = rounded(M.astype(np.float64), vtype)
        with fd.Spmm(dm, vtype) as op:
            y = op.run(torch.as_tensor(x).cuda())
            again = op.run(torch.as_tensor(x).cuda())
        assert torch.equal(y, again)
        want, mag = D.T @ x.astype(np.float64), np.abs(D).T @ np.abs(x.astype(np.float64))
        n = (D != 0).sum(0)[:, None]
        assert np.all(np.abs(y.cpu().numpy() - want) <= (n + 2) * U * mag), (k, vtype)


@pytest.mark.parametrize("k", [127, 129, 131, 255, 257, 515])
def test_product_of_odd_numbers_of_vectors_around_128(torch_cuda, k):
    """Beyond 128 vectors a wavefront takes one column at a time, also where k is no multiple of four."""
    test_product_over_lane_arrangements(torch_cuda, k)


@pytest.mark.parametrize("k", [65, 66, 127, 129, 131, 191, 255, 257, 515])
def test_product_of_odd_numbers_of_vectors(torch_cuda, k):
    """Beyond 64 vectors, where k is no multiple of four, a lane takes two or four vectors 64 apart and columns
    without entries are written in one run; also into memory that is not aligned to 16 bytes."""
    test_product_over_lane_arrangements(torch_cuda, k)
    torch = torch_cuda
    rng = np.random.default_rng(k)
    R, cols = 40, 1500
    off, c, v = random_rows(rng, R, cols, 0.01)
    keep = (c < 300) | (c >= 700)  # 400 columns without entries
    off = np.concatenate([[0], np.cumsum(keep)])[off]
    mats = [(off, c[keep], v[keep])]
    x = rng.uniform(-1.0, 1.0, (R, k)).astype(np.float32)
    xd = torch.as_tensor(x).cuda()
    with fd.Spmm(dose_mat(torch, cols, mats)) as op:
        y = op.run(xd).cpu().numpy()
        buf = torch.full((cols * k + 2,), -7.0, device="cuda")
        _lib.call("fd_spmm_run", op._h, C.c_void_p(xd.data_ptr()), k, C.c_void_p(buf[1:].data_ptr()), None)
        shifted = buf.cpu().numpy()
    D = dense(mats, cols)
    want, mag = D.T @ x.astype(np.float64), np.abs(D).T @ np.abs(x.astype(np.float64))
    assert np.all(np.abs(y - want) <= ((D != 0).sum(0)[:, None] + 2) * U * mag)
    assert np.array_equal(shifted[1:-1].reshape(cols, k), y) and shifted[0] == shifted[-1] == -7.0


@pytest.mark.parametrize("vtype", [fd.FD_VAL_BF16, fd.FD_VAL_FP16])
@pytest.mark.parametrize("x1", [1e10, float("inf"), float("nan"), 0.0])
def test_one_vector_beyond_the_float_range(torch_cuda, vtype, x1):
    """A row whose maximum times x is not finite while its other entries' products are: one vector gives
    what the same vector beside a second one gives (columns of at most three entries: same order)."""
    torch = torch_cuda
    cols = 5000
    rng = np.random.default_rng(3)
    v = rng.uniform(1e25, 1e27, (3, cols)).astype(np.float32)
    v[:, 100] = 1e30
    off = np.arange(4) * cols
    c = np.tile(np.arange(cols, dtype=np.int64), 3)
    with fd.Spmm(dose_mat(torch, cols, [(off, c, v.reshape(-1))]), vtype) as op:
        x = torch.tensor([[1.0], [x1], [1e-3]], device="cuda")
        one = op.run(x).cpu().numpy()[:, 0]
        two = op.run(torch.cat([x, torch.ones_like(x)], 1).contiguous()).cpu().numpy()[:, 0]
    if x1 == 1e10:
        assert np.isinf(two[100]) and np.isfinite(np.delete(two, 100)).all()
    if x1 == 0.0:  # the table's path: q (s x) against (q s) x, three terms of one sign
        assert np.all(np.abs(one.astype(np.float64) - two) <= 8 * U * np.abs(two))
    else:
        assert np.array_equal(one, two, equal_nan=True)


@pytest.mark.parametrize("R,cols", [(47, 192 * 2048 - 1), (48, 192 * 2048 - 1), (48, 192 * 2048), (2, 2 * 8192 + 1),
                                    (2, 2 * 8192), (1500, 511), (1500, 513), (70, 300 * 2048 + 5)])
def test_tile_widths(torch_cuda, R, cols):
    """Tiles of 512 columns below 192 x 2048 columns and with a row for 8192 of them at least, of 2048 otherwise:
    both sides of the lines, rows with every column of some tiles, against the general path, bit for bit."""
    torch = torch_cuda
    rng = np.random.default_rng([R, cols])
    rows = []
    for r in range(R):
        start = int(rng.integers(0, max(1, cols - 3000)))
        long = np.arange(start, min(cols, start + int(rng.integers(1, 3000)))) if r % 9 == 1 else np.zeros(0, np.int64)
        rows.append(np.unique(np.concatenate([rng.integers(0, cols, 900), long, [0, cols - 1]])))
    off = np.concatenate([[0], np.cumsum([len(c) for c in rows])])
    c = np.concatenate(rows).astype(np.int64)
    v = rng.uniform(0.01, 1.0, len(c)).astype(np.float32)
    back = np.concatenate([np.arange(off[r], off[r + 1])[::-1] for r in range(R)])
    x = torch.rand((R, 3), device="cuda")
    for vtype in (fd.FD_VAL_F32, fd.FD_VAL_BF16, fd.FD_VAL_FP16):
        y = []
        for m in ((off, c, v), (off, c[back], v[back])):
            with fd.Spmm(dose_mat(torch, cols, [m]), vtype) as op:
                y.append(op.run(x).cpu().numpy())
        assert np.array_equal(*y) and (y[0][0] > 0).all() and (y[0][-1] > 0).all()


@pytest.mark.parametrize("R,cols,fill", [(2, (1 << 19) - 1, 1.0), (2, 1 << 19, 1.0), (2, 1 << 19, 0.7),
                                         (255, (1 << 17) + 3, 0.02), (255, (1 << 17) - 3, 0.02),
                                         (255, (1 << 17) + 3, 0.006), (4096, 1 << 17, 0.009), (4097, 1 << 17, 0.009)])
def test_one_vector_and_16_bit_values_in_large_volumes(torch_cuda, R, cols, fill):
    """The products of scales and vector lie in LDS from 2^17 columns on where the columns hold enough entries:
    both sides of each line."""
    torch = torch_cuda
    rng = np.random.default_rng([R, cols, int(1000 * fill)])
    n = round(fill * cols)
    c = np.concatenate([np.sort((int(rng.integers(cols)) + np.arange(n)) % cols) for _ in range(R)])
    v = rng.uniform(0.01, 1.0, R * n).astype(np.float32)
    x = rng.uniform(-1.0, 1.0, (R, 1)).astype(np.float32)
    row = np.repeat(np.arange(R), n)
    dm = dose_mat(torch, cols, [(np.arange(R + 1) * n, c, v)])
    for vtype in (fd.FD_VAL_BF16, fd.FD_VAL_FP16):
        stored = rounded(v.reshape(R, n).astype(np.float64), vtype).reshape(-1)
        with fd.Spmm(dm, vtype) as op:
            y = op.run(torch.as_tensor(x).cuda()).cpu().numpy()[:, 0]
        term = stored * x[row, 0].astype(np.float64)
        want, mag = (np.bincount(c, w, cols) for w in (term, np.abs(term)))
        assert np.all(np.abs(y - want) <= (np.bincount(c, minlength=cols) + 3) * U * mag), vtype


@pytest.mark.parametrize("vtype", [fd.FD_VAL_BF16, fd.FD_VAL_FP16])
@pytest.mark.parametrize("x1", [1e10, float("inf"), float("nan"), 0.0])
def test_one_vector_beyond_the_float_range_in_large_volumes(torch_cuda, vtype, x1):
    """As with few columns, where the products of scales and vector lie in LDS."""
    torch = torch_cuda
    cols = (1 << 19) + 5
    rng = np.random.default_rng(3)
    v = rng.uniform(1e25, 1e27, (3, cols)).astype(np.float32)
    v[:, 100] = 1e30
    c = np.tile(np.arange(cols, dtype=np.int64), 3)
    with fd.Spmm(dose_mat(torch, cols, [(np.arange(4) * cols, c, v.reshape(-1))]), vtype) as op:
        x = torch.tensor([[1.0], [x1], [1e-3]], device="cuda")
        one = op.run(x).cpu().numpy()[:, 0]
        two = op.run(torch.cat([x, torch.ones_like(x)], 1).contiguous()).cpu().numpy()[:, 0]
    if x1 == 1e10:
        assert np.isinf(two[100]) and np.isfinite(np.delete(two, 100)).all()
    if x1 == 0.0:  # the table's path: q (s x) against (q s) x, three terms of one sign
        assert np.all(np.abs(one.astype(np.float64) - two) <= 8 * U * np.abs(two))
    else:
        assert np.array_equal(one, two, equal_nan=True)
