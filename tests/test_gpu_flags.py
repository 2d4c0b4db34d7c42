"""Device beamlet flags against the host's, bit for bit, where the mask's bounding box and the depth
range cut from it can go wrong: single texels at corners and edges, one-texel-thick planes, an empty and a
full mask, masks at every byte alignment, odd dimensions, beams along the axes (needs an MI355X)."""
import numpy as np
import pytest

import fastdose_amd as fd
from fastdose_amd import synth

pytestmark = pytest.mark.gpu

DIM = (37, 29, 23)


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def masks():
    X, Y, Z = DIM
    out = {}
    for name, at in {"corner": (0, 0, 0), "far corner": (Z - 1, Y - 1, X - 1), "edge": (Z // 2, 0, X - 1),
                     "middle": (Z // 2, Y // 2, X // 2)}.items():
        m = np.zeros((Z, Y, X), np.uint8)
        m[at] = 1
        out[name] = m
    plane = np.zeros((Z, Y, X), np.uint8)
    plane[:, Y // 3, :] = 255
    out["plane"] = plane
    two = np.zeros((Z, Y, X), np.uint8)
    two[1, 2, 3] = two[Z - 2, Y - 3, X - 4] = 7
    out["two texels"] = two
    out["empty"] = np.zeros((Z, Y, X), np.uint8)
    out["full"] = np.ones((Z, Y, X), np.uint8)
    out["speckle"] = (np.random.default_rng(1).random((Z, Y, X)) < 0.002).astype(np.uint8)
    return out


@pytest.mark.parametrize("name", list(masks()))
def test_flags_equal_the_host(torch_cuda, name):
    torch = torch_cuda
    m = masks()[name]
    vol = synth.make_volume(DIM, 0.25)
    rng = np.random.default_rng(sum(map(ord, name)))
    iso = [0.25 * d / 2 for d in DIM]
    angles = [(0, 0, 0), (90, 0, 0), (180, 0, 0), (270, 90, 0), (90, 90, 0)] + \
        [tuple(rng.uniform(0, 360, 3)) for _ in range(12)]
    bundles = []
    for a in angles:
        at = [c + float(rng.uniform(-2, 2)) for c in iso]
        bundles.append(synth.make_bundle(at, a, fluence_dim=int(rng.integers(1, 24)), beamlet_size=0.4,
                                         long_spacing=float(rng.choice([0.25, 0.1, 0.7]))))
    want = []
    for b in bundles:
        try:
            want.append(fd.beamlet_flag_init(b, m, vol))
        except fd.FastDoseError:
            want.append(np.zeros(b.fluence_dim[0] ** 2, np.uint8))
    with fd.Context(vol, np.ones(DIM[::-1], np.float32), synth.synthetic_spectrum(1), synth.synthetic_kernel(1)) as ctx:
        for shift in (0, 1, 7, 15):
            buf = torch.zeros(m.size + 16, dtype=torch.uint8, device="cuda")
            buf[:shift] = 1            # texels beside the mask are not part of it
            buf[shift + m.size:] = 1
            buf[shift:shift + m.size] = torch.from_numpy(m.reshape(-1)).cuda()
            got = ctx.beamlet_flags(buf[shift:], bundles)
            for w, g in zip(want, got):
                assert np.array_equal(w, g)
    if name in ("full", "plane"):
        assert any(w.any() for w in want)


@pytest.mark.parametrize("voxel", [0.25, 0.3, float(np.uint32(0x3E7FFFFF).view(np.float32))])
@pytest.mark.parametrize("dim", [(1, 29, 23), (2, 1, 23), (3, 29, 1), (24, 17, 2)])
def test_flags_in_thin_volumes(torch_cuda, dim, voxel):
    """Volumes one to three voxels wide, where the pair of texels read along x does not fit or is the whole
    row, and voxel sizes whose division is exact, corrected, and (all ones in the significand) done as a
    division; beams shifted so that sample points fall on texel boundaries among others."""
    torch = torch_cuda
    vol = synth.make_volume(dim, voxel)
    rng = np.random.default_rng(list(dim))
    masks = [(rng.random(dim[::-1]) < f).astype(np.uint8) for f in (0.02, 0.3)] + [np.ones(dim[::-1], np.uint8)]
    iso = [voxel * d / 2 for d in dim]
    bundles = []
    for a in [(0, 0, 0), (90, 0, 0), (90, 90, 0)] + [tuple(rng.uniform(0, 360, 3)) for _ in range(9)]:
        at = [c + float(rng.integers(-2, 3)) * voxel / 2 for c in iso]
        bundles.append(synth.make_bundle(at, a, fluence_dim=int(rng.integers(1, 12)), beamlet_size=3 * voxel,
                                         long_spacing=voxel))
    some = 0
    with fd.Context(vol, np.ones(dim[::-1], np.float32), synth.synthetic_spectrum(1), synth.synthetic_kernel(1)) as ctx:
        for m in masks:
            got = ctx.beamlet_flags(torch.from_numpy(m.reshape(-1)).cuda(), bundles)
            for b, g in zip(bundles, got):
                try:
                    w = fd.beamlet_flag_init(b, m, vol)
                except fd.FastDoseError:
                    w = np.zeros(b.fluence_dim[0] ** 2, np.uint8)
                assert np.array_equal(w, g)
                some += int(w.any())
    assert some > 0


@pytest.mark.parametrize("name", list(masks()))
def test_flags_with_and_without_the_box(torch_cuda, name):
    """One beamlet and 16 of them (fewer sample points than it pays to look for the mask's box) and 30 beams of
    400 (more): the host's flags."""
    torch = torch_cuda
    m = masks()[name]
    vol = synth.make_volume(DIM, 0.25)
    rng = np.random.default_rng(sum(map(ord, name)) + 1)
    at = [0.25 * (d / 2 + float(rng.uniform(-4, 4))) for d in DIM]
    angles = [(0, 0, 0), (90, 0, 0)] + [tuple(rng.uniform(0, 360, 3)) for _ in range(4)]
    with fd.Context(vol, np.ones(DIM[::-1], np.float32), synth.synthetic_spectrum(1), synth.synthetic_kernel(1)) as ctx:
        for fluence, copies in ((1, 1), (4, 1), (20, 5)):
            bundles = [synth.make_bundle(at, a, fluence_dim=fluence, beamlet_size=0.4, long_spacing=0.25) for a in angles]
            want = [fd.beamlet_flag_init(b, m, vol) for b in bundles]
            points = sum(9 * fd.calc_range(beam_of(b), vol).long_dim * fluence ** 2 for b in bundles) * copies
            assert (points > 200_000 + m.size // 64) == (copies == 5)
            for shift in (0, 5):
                buf = torch.zeros(m.size + 16, dtype=torch.uint8, device="cuda")
                buf[shift:shift + m.size] = torch.from_numpy(m.reshape(-1)).cuda()
                got = ctx.beamlet_flags(buf[shift:], bundles * copies)
                for w, g in zip(want * copies, got):
                    assert np.array_equal(w, g)


def beam_of(bundle):
    beam = fd.Beam()
    for f in ("isocenter", "angles", "beamlet_size"):
        for i, v in enumerate(getattr(bundle, f)):
            getattr(beam, f)[i] = v
    beam.fmap_size[0], beam.fmap_size[1] = bundle.fluence_dim[0], bundle.fluence_dim[1]
    beam.sad, beam.long_spacing = bundle.sad, bundle.long_spacing
    return beam

