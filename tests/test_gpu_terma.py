"""Terma's density records on both sides of 4 GiB (needs an MI355X): 32-bit record offsets below,
64-bit ones from there on.  The same beamlets through the same voxels, in the corner of two volumes
whose other voxels are empty, sample the same densities.  The volumes have diagonals of the same length
(30^2 + 36^2 + 885^2 = 509^2 + 512^2 + 514^2), so their contexts tabulate the spectrum alike: the outputs
are the same bits.
"""
import numpy as np
import pytest

import fastdose_amd as fd
from fastdose_amd import synth

from gpu_util import beamlets_of, log

pytestmark = pytest.mark.gpu
NPIX = 256


@pytest.mark.parametrize("options", [0, fd.FD_OPT_RPL_FP64_ALL])
def test_record_offsets(options):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    cfg = synth.small_config(seed=17, dim=(23, 26, 22), fluence_dim=3, angles=(35.0, 20.0, 0.0))
    beams, flu = beamlets_of(cfg)
    stride = max(b.long_dim for b in beams) * NPIX
    flu_d = torch.from_numpy(np.ascontiguousarray(flu, dtype=np.float32)).cuda()
    got = []
    for dim in ((30, 36, 885), (509, 512, 514)):
        density = np.zeros(dim[::-1], dtype=np.float32)
        density[:22, :26, :23] = np.asarray(cfg.density, dtype=np.float32).reshape(22, 26, 23)
        vol = synth.make_volume(dim, cfg.volume.voxel_size[0])
        assert list(vol.voxel_size) == list(cfg.volume.voxel_size)
        log(f"terma in {dim}, options {options}")
        with fd.Context(vol, density, cfg.spectrum, cfg.kernel, options=options) as ctx:
            T = torch.zeros(len(beams) * stride, device="cuda")
            R = torch.zeros_like(T)
            ctx.terma(beams, flu_d, T, R, stride)
            torch.cuda.synchronize()
            got.append((T.cpu().numpy(), R.cpu().numpy()))
    assert got[0][0].max() > 0 and got[0][1].max() > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
