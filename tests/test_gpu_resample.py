"""Room for the resampler's output and staging (needs an MI355X): outputs of exactly the entries found, one
less, none and the estimate; a staging area that the estimate makes too small (more candidates than the
frustums suggest, so the values are computed twice); a result far below the estimate."""
import ctypes as C

import numpy as np
import pytest

import fastdose_amd as fd
from fastdose_amd import _lib, synth

from gpu_util import beamlets_of, log

pytestmark = pytest.mark.gpu
NPIX = 256


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.fixture()
def case(torch_cuda):
    torch = torch_cuda
    cfg = synth.small_config(seed=29, dim=(31, 27, 30), fluence_dim=4, angles=(25.0, 40.0, 0.0))
    beams, _ = beamlets_of(cfg)
    stride = max(b.long_dim for b in beams) * NPIX
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    dose = torch.rand(len(beams) * stride, device="cuda", generator=g)

    def context():
        return fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel)

    return context, beams, dose, stride


def rows(result):
    return [t.cpu().numpy() for t in result]


def test_output_room(torch_cuda, case):
    torch = torch_cuda
    context, beams, dose, stride = case
    with context() as ctx:
        want = rows(ctx.resample_csr(beams, dose, stride))
        nnz, n = len(want[1]), len(beams)
        assert nnz > 0
        cap = C.c_uint64()
        _lib.call("fd_resample_capacity", ctx._h, beams, n, C.byref(cap))
        for room in (0, nnz - 1, nnz, nnz + 1, max(cap.value, nnz)):
            log(f"resample into {room} of {nnz}")
            off = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
            cols = torch.full((room + 8,), -1, dtype=torch.int64, device="cuda")
            vals = torch.full((room + 8,), -1.0, device="cuda")
            csr = fd.CSR(0, 0, room, off.data_ptr(), cols.data_ptr() if room else None,
                         vals.data_ptr() if room else None)
            rc = _lib.load().fd_resample_csr(ctx._h, beams, n, C.c_void_p(dose.data_ptr()), stride, 2.0,
                                             C.byref(csr), None)
            torch.cuda.synchronize()
            assert csr.nnz == nnz and csr.rows == n
            assert rc == (_lib.FD_OK if room >= nnz else _lib.FD_ERR_CAPACITY)
            assert np.array_equal(off.cpu().numpy(), want[0]) or rc != _lib.FD_OK
            if rc == _lib.FD_OK:
                assert np.array_equal(cols[:nnz].cpu().numpy(), want[1])
                assert np.array_equal(vals[:nnz].cpu().numpy(), want[2])
            assert (cols[room:] == -1).all() and (vals[room:] == -1.0).all()  # nothing beyond the room


def test_staging_too_small(torch_cuda, case):
    """A context that has seen one beamlet of sixteen inside the volume expects few candidates per frustum;
    with all of them inside, its staging overflows and the values are computed a second time."""
    context, beams, dose, stride = case
    with context() as ctx:
        want = rows(ctx.resample_csr(beams, dose, stride))
    away = fd.beam_array(list(beams))
    for b in list(away)[1:]:
        for d in range(3):
            b.source[d] += 1000.0
    cap = C.c_uint64()
    with context() as ctx:
        log("resample, most beamlets beside the volume")
        few = rows(ctx.resample_csr(away, dose, stride))
        assert np.array_equal(few[1], want[1][:want[0][1]]) and np.array_equal(few[2], want[2][:want[0][1]])
        _lib.call("fd_resample_capacity", ctx._h, beams, len(beams), C.byref(cap))
        assert cap.value < len(want[1])
        log("resample, staging too small")
        got = rows(ctx.resample_csr(beams, dose, stride))
        _lib.call("fd_resample_capacity", ctx._h, beams, len(beams), C.byref(cap))
        assert cap.value >= len(want[1])
        log("resample, staging known")
        again = rows(ctx.resample_csr(beams, dose, stride))
    for a, b, c in zip(want, got, again):
        assert np.array_equal(a, b) and np.array_equal(a, c)


def test_result_far_below_the_estimate(torch_cuda, case):
    torch = torch_cuda
    context, beams, dose, stride = case
    with context() as ctx:
        full = rows(ctx.resample_csr(beams, dose, stride))
        one = torch.zeros_like(dose)
        one[:NPIX] = dose[:NPIX]  # the first slice of the first beamlet
        off, cols, vals = ctx.resample_csr(beams, one, stride)
        none = rows(ctx.resample_csr(beams, torch.zeros_like(dose), stride))
    assert 0 < len(cols) < len(full[1])
    assert cols.untyped_storage().nbytes() <= 8 * (2 * len(cols) + 1024)
    assert off[1] == len(cols) and (off[1:] == len(cols)).all() and (vals > 0).all()
    assert len(none[1]) == len(none[2]) == 0 and not none[0].any()


def test_estimate_beyond_the_device(torch_cuda, case, monkeypatch):
    """An estimate for which there is no memory: the result comes from a sizing call and arrays of its size."""
    context, beams, dose, stride = case
    with context() as ctx:
        want = rows(ctx.resample_csr(beams, dose, stride))
        real = fd.host.call

        def call(name, *args):
            real(name, *args)
            if name == "fd_resample_capacity":
                args[-1]._obj.value = 1 << 45
            return _lib.FD_OK

        monkeypatch.setattr(fd.host, "call", call)
        got = rows(ctx.resample_csr(beams, dose, stride))
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


def test_failed_allocation_is_reported_once(torch_cuda):
    """A matrix whose operator would need 2 TB: the call fails, and the next launches are not blamed for it."""
    torch = torch_cuda
    with pytest.raises(fd.FastDoseError, match="out of memory"):
        fd.Spmm(fd.DoseMat(1 << 38))
    d = torch.ones((3, 5), device="cuda")
    off, cols, vals = fd.host.dense_to_csr(d)
    assert off.tolist() == [0, 5, 10, 15] and cols.tolist() == list(range(5)) * 3 and (vals == 1.0).all()
