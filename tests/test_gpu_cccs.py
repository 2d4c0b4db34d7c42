"""CCCS workgroups of every size of the march and table kernels (needs an MI355X).

A workgroup has one wavefront per azimuth, and one more in the march kernel.  With less than four
wavefronts each slab is loaded when its slice starts, with four to seven a wavefront loads two groups
of the next slab ahead, from eight on one: the azimuth counts on both sides of these lines, against
the oracle at the tolerances of the other kernel shapes, and the table kernel against the march
kernel bit for bit.
"""
import numpy as np
import pytest

import fastdose_amd as fd
import oracle as orc
from fastdose_amd import synth

from gpu_util import beamlets_of, gpu_stages, log, same_matrix
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.mark.parametrize("n_phi", [1, 3, 4, 6, 7, 9])
@pytest.mark.parametrize("exact_g", [False, True])
def test_workgroup_sizes(torch_cuda, n_phi, exact_g):
    cfg = synth.small_config(seed=70 + n_phi, dim=(22, 26, 23), fluence_dim=2, angles=(40.0, -30.0, 15.0))
    cfg.kernel = synth.synthetic_kernel(1070 + n_phi, n_phi=n_phi)
    flag = fd.FD_OPT_EXACT_G if exact_g else 0
    beams, flu = beamlets_of(cfg)
    log(f"azimuths {n_phi} exact_g={exact_g}")
    with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel, options=flag) as ctx:
        g = gpu_stages(ctx, beams, flu, cfg.extent)
    check_against_oracle(cfg, beams, flu, g, range(len(beams)), flags=orc.EXACT_G if exact_g else 0)
    flags = [np.ones(4, dtype=np.uint8)]
    mats = []
    for how in (fd.FD_OPT_NO_TABLES, fd.FD_OPT_TABLES):
        with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel, options=flag | how) as ctx:
            mats.append(fd.dose_mat_construction(ctx, cfg.bundles, flags, cfg.extent, batched=True))
    assert mats[0].info() == mats[1].info() and mats[0].info()[2] > 0
    assert same_matrix(mats[0].matrix(0), mats[1].matrix(0))


@pytest.mark.parametrize("n_phi", [8, 10])
@pytest.mark.parametrize("exact_g", [False, True])
def test_split_widest_cone(torch_cuda, n_phi, exact_g):
    """Up to 51 beamlets (four forward cones: 255 workgroups) the widest cone's azimuths take two workgroups
    each; 56 beamlets in one call (no split) and in calls of 51, 4 and 1 (all split): the same bits, also
    with a slice spacing at which the march of azimuth 0 skips slices and others take several chunks."""
    cfg = synth.small_config(seed=95 + n_phi, dim=(30, 26, 28), fluence_dim=8, angles=(20.0, 15.0, 0.0))
    cfg.kernel = synth.synthetic_kernel(1095, n_phi=n_phi)
    all_beams, flu = beamlets_of(cfg)
    for spacing in (1.0, 6.0, 0.2):
        beams = fd.beam_array(list(all_beams)[:56])
        for b in beams:
            b.long_spacing *= spacing
            b.long_dim = max(1, int(np.ceil(b.long_dim / spacing)))
        log(f"split cone, {n_phi} azimuths, exact_g={exact_g}, slice spacing x {spacing}")
        options = fd.FD_OPT_EXACT_G if exact_g else 0
        with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel, options=options) as ctx:
            dose = gpu_stages(ctx, beams, flu[:56], cfg.extent)["dose"]
            k = 0
            for a, b in ((0, 51), (51, 55), (55, 56)):
                for d in gpu_stages(ctx, fd.beam_array(beams[a:b]), flu[a:b], cfg.extent)["dose"]:
                    L = beams[k].long_dim
                    assert np.array_equal(d[:L], dose[k, :L]) and d[:L].max() > 0
                    k += 1


def test_few_and_many_workgroups(torch_cuda):
    """144 beamlets (four forward cones: 576 workgroups) in one call and in calls of 128 and 16: the
    instances for few and for many workgroups, the first at its largest."""
    cfg = synth.small_config(seed=91, dim=(30, 26, 28), fluence_dim=12, angles=(20.0, 15.0, 0.0))
    beams, flu = beamlets_of(cfg)
    assert len(beams) == 144
    for options in (0, fd.FD_OPT_EXACT_G):
        log(f"few and many workgroups, options {options}")
        with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel, options=options) as ctx:
            dose = gpu_stages(ctx, beams, flu, cfg.extent)["dose"]
            parts = [gpu_stages(ctx, fd.beam_array(beams[a:b]), flu[a:b], cfg.extent)["dose"]
                     for a, b in ((0, 128), (128, 144))]
        k = 0
        for part in parts:
            for d in part:
                L = beams[k].long_dim
                assert np.array_equal(d[:L], dose[k, :L]) and d[:L].max() > 0
                k += 1


def test_split_partials_stay_small(torch_cuda):
    """A split cone takes more partial volumes (nine instead of four here), but not beyond 512 MiB: one
    beamlet of 50 000 slices is split (440 MiB), one of 60 000 (527) is not; the slices they share are the
    same bits."""
    torch = torch_cuda
    cfg = synth.small_config(seed=77, dim=(22, 26, 23), fluence_dim=1, angles=(20.0, 15.0, 0.0))
    cfg.kernel = synth.synthetic_kernel(1077, n_phi=8)
    beams, _ = beamlets_of(cfg)
    beams = fd.beam_array(list(beams)[:1])
    depth = beams[0].long_spacing * beams[0].long_dim
    slice_floats = 256
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    T = torch.rand(60000 * slice_floats, device="cuda", generator=g)
    R = torch.rand(60000 * slice_floats, device="cuda", generator=g) + 0.5
    dose, taken = [], []
    for L in (50000, 60000):
        beams[0].long_dim, beams[0].long_spacing = L, depth / 60000
        D = torch.zeros(L * slice_floats, device="cuda")
        log(f"split partials, {L} slices")
        with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel) as ctx:
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info()[0]
            ctx.cccs(beams, T[:D.numel()], R[:D.numel()], D, D.numel())
            torch.cuda.synchronize()
            taken.append(free - torch.cuda.mem_get_info()[0])
        dose.append(D)
    assert torch.equal(dose[0], dose[1][:dose[0].numel()]) and float(dose[0].max()) > 0
    assert taken[0] > 8 * 50000 * slice_floats * 4      # the split's volumes
    assert taken[1] < 5 * 60000 * slice_floats * 4


def test_no_split_volumes_beside_march_tables(torch_cuda):
    """A served batch of 16 beamlets: with march tables the widest cone is not split, and the batch counts
    five volumes less."""
    cfg = synth.small_config(seed=78, dim=(30, 26, 28), fluence_dim=4, angles=(20.0, 15.0, 0.0))
    cfg.kernel = synth.synthetic_kernel(1078, n_phi=8)
    beams, flu = beamlets_of(cfg)
    peak, mats = [], []
    with fd.Context(cfg.volume, cfg.density, cfg.spectrum, cfg.kernel) as ctx:
        for how in (fd.FD_OPT_NO_TABLES, fd.FD_OPT_TABLES):
            log(f"served batch, options {how}")
            with fd.Server(ctx, n_slots=1, options=how) as server:
                mats.append(server.fetch(server.submit(beams, flu, [len(beams)])))
                peak.append(server.stats()["peak_inflight_bytes"])
    assert peak[0] - peak[1] == 5 * 4 * 256 * sum(b.long_dim for b in beams)
    assert same_matrix(mats[0].matrix(0), mats[1].matrix(0))
