"""Context.resample_csr where the device has no room for the estimate (CPU: a stand-in for the library whose
memory, shared with the output arrays, is counted in entries): whatever fits with arrays of the exact size is
still returned, and an allocation that failed for another reason is still an error."""
import ctypes as C

import numpy as np
import pytest
import torch

import fastdose_amd as fd
from fastdose_amd import _lib, host

ESTIMATE, NNZ = 4096, 1500


class Card:
    """The library's two calls and torch.empty on a card with room for `entries` entries of arrays and
    `staging` entries of the library's scratch, both from the same memory."""

    def __init__(self, memory, failure=b"hipMalloc: out of memory"):
        self.memory, self.failure, self.held, self.error, self.rooms = memory, failure, {}, b"", []
        self.real_empty = torch.empty

    def used(self):
        import gc

        gc.collect()
        return sum(n for r, n in self.held.values() if r() is not None)

    def empty(self, n, dtype=None, device=None):
        import weakref

        t = self.real_empty(n, dtype=dtype)
        if dtype == torch.int64 and n > 64:  # the columns stand for columns and values
            if self.used() + n > self.memory:
                raise torch.OutOfMemoryError("out of memory")
            self.held[id(t)] = (weakref.ref(t), n)
        return t

    def fd_resample_csr(self, ctx, arr, n, dose, stride, extent, csr, stream):
        csr = csr._obj
        self.rooms.append(csr.capacity)
        if self.used() + ESTIMATE > self.memory:  # the staging does not fit beside the arrays
            self.error = self.failure
            return _lib.FD_ERR_HIP
        csr.nnz = NNZ
        off = np.ctypeslib.as_array(C.cast(csr.offsets, C.POINTER(C.c_int64)), (n + 1,))
        off[:] = [0, 1000, NNZ]
        if csr.capacity < NNZ or not csr.columns or not csr.values:
            return _lib.FD_ERR_CAPACITY
        np.ctypeslib.as_array(C.cast(csr.columns, C.POINTER(C.c_int64)), (NNZ,))[:] = np.arange(NNZ) * 3
        np.ctypeslib.as_array(C.cast(csr.values, C.POINTER(C.c_float)), (NNZ,))[:] = np.arange(NNZ) + 0.5
        return _lib.FD_OK

    def fd_last_error(self):
        return self.error

    def call(self, name, ctx, arr, n, *rest):
        if name == "fd_resample_capacity":
            rest[0]._obj.value = ESTIMATE
            return _lib.FD_OK
        return _lib.check(getattr(self, name)(ctx, arr, n, *rest), name)


def resample(monkeypatch, card):
    monkeypatch.setattr(_lib, "load", lambda: card)
    monkeypatch.setattr(host, "load", lambda: card)
    monkeypatch.setattr(host, "call", card.call)
    monkeypatch.setattr(torch, "empty", card.empty)
    ctx = host.Context.__new__(host.Context)
    ctx._h = None
    return ctx.resample_csr((fd.Beam * 2)(), torch.zeros(512), 256)


# arrays and staging of the estimate; staging and exact arrays only; the same to the entry; and less room
# for arrays of the estimate than for nothing
@pytest.mark.parametrize("memory", [3 * ESTIMATE, 2 * ESTIMATE - 1, ESTIMATE + NNZ + 600, ESTIMATE + NNZ])
def test_result_fits_as_with_exact_arrays(monkeypatch, memory):
    card = Card(memory)
    off, cols, vals = resample(monkeypatch, card)
    assert off.tolist() == [0, 1000, NNZ]
    assert torch.equal(cols, torch.arange(NNZ) * 3) and torch.equal(vals, torch.arange(NNZ) + 0.5)
    assert card.rooms[0] == ESTIMATE or memory < ESTIMATE
    if memory >= 2 * ESTIMATE:
        assert len(card.rooms) == 1


def test_errors_stay_errors(monkeypatch):
    with pytest.raises((torch.OutOfMemoryError, fd.FastDoseError)):
        resample(monkeypatch, Card(ESTIMATE + NNZ - 1))
    card = Card(2 * ESTIMATE - 1, failure=b"resample values launch: invalid device function")
    with pytest.raises(fd.FastDoseError, match="invalid device function"):
        resample(monkeypatch, card)
    assert len(card.rooms) == 1
