"""The work this library is timed on: dose-matrix construction and what is done with the matrix.

A case is one call, or one short chain of calls, that a treatment-planning program makes through the
package's entry points.  Kinds:

    stages    Terma -> CCCS -> resampling of one beam's beamlets on device buffers
    terma, cccs, resample   one of the three stages alone
    matrix    DoseMat.add_beam of one beam of a 4pi plan, its CSR matrix fetched to the host
    plan      DoseMat.add_beams of several beams, the voxel-major operator built, D^T X of it
    serve     requests of 1-4 beams through a running Server, fetched into one matrix, then as plan
    product   D^T X on an operator that is in place (the optimiser's inner loop)
    dense     dense -> CSR conversion of one beam's dose rows
    flags     beamlet / PTV intersection flags of many beams

The single stages take synthetic pencil beams whose geometry this file computes itself, so that
exact() can follow the same definitions in 64 bits without the library.  A case fixes where its beams
lie; the seed fills in the medium, the tables, the fluence and the operands.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import fastdose_amd as fd
from fastdose_amd import _lib, host, synth

VOXEL = 0.25          # cm, every configuration of the repository
SAD = 100.0
NPIX = 256            # 16 x 16 BEV pixels per beamlet
STAGES = ("stages", "terma", "cccs", "resample")
VALUE_TYPES = {"f32": fd.FD_VAL_F32, "bf16": fd.FD_VAL_BF16, "fp16": fd.FD_VAL_FP16}


def listed():
    return [
        # four beamlets in a 24^3 box: the smallest beam of the tests; launches and latency only
        dict(name="stages-box24", kind="stages", x=24, y=24, z=24, side=2, phi=8, medium="slab", exact_g=False),
        # the 64^3 water phantom, one 8 x 8 beam
        dict(name="stages-water64", kind="stages", x=64, y=64, z=64, side=8, phi=8, medium="water", exact_g=False),
        # the 128^3 slab phantom, one 16 x 16 beam, stage by stage
        dict(name="terma-slab128", kind="terma", x=128, y=128, z=128, side=16, phi=8, medium="slab", rpl64=False),
        dict(name="cccs-slab128", kind="cccs", x=128, y=128, z=128, side=16, phi=8, medium="slab", exact_g=False),
        dict(name="resample-slab128", kind="resample", x=128, y=128, z=128, side=16, phi=8, medium="slab"),
        # one beam of the 4pi plan on the 200 x 200 x 160 body, one call per beam as in the reference's loop
        dict(name="matrix-body200", kind="matrix", x=200, y=200, z=160, beams=1, fluence=20),
        # a 20-beam plan on the same body: all beams in one call, then the optimiser's operator and a first dose
        dict(name="plan-body200", kind="plan", x=200, y=200, z=160, beams=20, fluence=20, type="f32", k=1),
        # the serving body: twelve beams in requests of 1-4 through a resident server, 16-bit operator
        dict(name="serve-body220", kind="serve", x=220, y=220, z=150, beams=12, fluence=20, type="bf16", k=4),
        # 256 fluence vectors through one slab beam's operator
        dict(name="product-f32-k256", kind="product", x=128, y=128, z=128, beams=1, rows=256, patch=8, type="f32",
             k=256),
        # one fluence vector through a 20-beam operator, 16-bit values: a step of the optimiser
        dict(name="product-bf16-k1", kind="product", x=200, y=200, z=160, beams=20, rows=133, patch=10, type="bf16",
             k=1),
        # the dense rows of the water beam
        dict(name="dense-water64", kind="dense", rows=64, cols=64 ** 3, fill=0.02),
        # every beam of the 180-beam plan against its target
        dict(name="flags-body200", kind="flags", x=200, y=200, z=160, beams=180, fluence=20),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["stages", "stages", "terma", "cccs", "resample", "matrix", "plan", "serve", "product",
                       "product", "dense", "flags"])
    if kind in STAGES:
        c = dict(kind=kind, x=log(20, 140), y=log(24, 160), z=log(20, 130), side=log(1, 14),
                 phi=rng.choice([8, 8, 8, 5, 12, 16]), medium=rng.choice(["slab", "slab", "water"]))
        if c["side"] > 2:  # the beam's field lies inside the volume
            for a in "xyz":
                c[a] = max(c[a], 4 * c["side"])
        if kind == "terma":
            c["rpl64"] = rng.random() < 0.3
        if kind in ("stages", "cccs"):
            c["exact_g"] = rng.random() < 0.25
        return c
    if kind in ("matrix", "plan", "serve"):
        c = dict(kind=kind, x=rng.randint(150, 220), y=rng.randint(150, 220), z=rng.randint(110, 160),
                 beams=1 if kind == "matrix" else log(2, 16), fluence=20)
        if kind != "matrix":
            c.update(type=rng.choice(["f32", "bf16", "fp16"]), k=log(1, 8))
        return c
    if kind == "product":
        c = dict(kind=kind, x=rng.randint(60, 200), y=rng.randint(60, 200), z=rng.randint(60, 160),
                 beams=log(1, 18), rows=log(7, 150), patch=rng.randint(6, 10), type=rng.choice(["f32", "bf16", "fp16"]))
        most = 4e8 / (c["x"] * c["y"] * c["z"])
        c["k"] = min(256, log(1, max(2, most)))
        return c
    if kind == "dense":
        cols = log(500, 128 ** 3)
        return dict(kind=kind, rows=log(1, max(2, min(400, 3e7 / cols))), cols=cols,
                    fill=round(math.exp(rng.uniform(math.log(0.003), math.log(0.5))), 4))
    return dict(kind=kind, x=rng.randint(100, 220), y=rng.randint(100, 220), z=rng.randint(80, 160),
                beams=log(1, 180), fluence=rng.choice([12, 16, 20]))


# ------------------------------------------------------------------ inputs


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed) % (1 << 31))
    return g


def _dims(case):
    return case["x"], case["y"], case["z"]


def _place(case):
    """Where a case's beams lie: the same for every seed."""
    return np.random.default_rng([case["x"], case["y"], case["z"], case.get("side", 0), case.get("beams", 0)])


def _rotation(gantry, couch, coll=0.0):
    """BEV -> PVCS matrix: a turn of -(couch + coll) about y, then of gantry about the couch-turned z axis."""

    def rodrigues(r, t):
        s, c = math.sin(t), math.cos(t)
        k = np.array([[0, -r[2], r[1]], [r[2], 0, -r[0]], [-r[1], r[0], 0]])
        return c * np.eye(3) + s * k + (1 - c) * np.outer(r, r)

    axis = np.array([math.sin(-couch), 0.0, math.cos(-couch)])
    return rodrigues(axis, gantry) @ rodrigues(np.array([0.0, 1.0, 0.0]), -(couch + coll))


def _spectrum(rng):
    """Twelve bins of 0.5 MeV with power-law attenuation, random decreasing weights."""
    energy = 0.5 + 0.5 * np.arange(12)
    w = np.sort(rng.uniform(0.0, 1.0, 12))[::-1]
    return tuple(np.asarray(v, np.float32) for v in (energy, w / w.sum(), 0.0707 * energy ** -0.523))


def _kernel(rng, n_phi):
    """Eight zenith cones of 22.5 degrees: (A, a, B, b) and mid angle of each, and the azimuths."""
    n = 8
    edge = (np.arange(n + 1) * (math.pi / n)).astype(np.float32)
    table = dict(A=np.sort(rng.uniform(0.5, 2.2, n))[::-1], a=rng.uniform(2.0, 8.0, n), B=rng.uniform(1e-3, 2.5e-2, n),
                 b=rng.uniform(0.05, 0.11, n), begin=edge[:-1], end=edge[1:], mid=(edge[:-1] + edge[1:]) / 2,
                 phi=(np.arange(n_phi) + 0.5) * (2 * math.pi / n_phi))
    return {k: np.asarray(v, np.float32) for k, v in table.items()}


def _slab_density(dims, medium, rng):
    X, Y, Z = dims
    if medium == "water":
        return np.ones((Z, Y, X), np.float32)
    cut = np.cumsum(rng.dirichlet([4.0, 4.0, 2.0, 4.0]) * Y)[:3]
    layer = np.array([1.0, 0.25, 1.8, 1.0], np.float32)[np.searchsorted(cut, np.arange(Y), side="right")]
    return np.ascontiguousarray(np.broadcast_to(layer[None, :, None], (Z, Y, X)))


def _pencils(case, seed):
    """One beam of side x side pencil beamlets, 5 mm apart, through the volume's centre, as numbers: the
    fields of a Beam (FP32), the density, the spectrum and the kernel table."""
    rng, place = np.random.default_rng(seed), _place(case)
    dims = _dims(case)
    side = case["side"]
    angles = np.radians([place.uniform(10.0, 60.0), place.uniform(5.0, 45.0), 0.0]).astype(np.float32)
    M = _rotation(*map(float, angles))
    centre = np.array(dims) * VOXEL * 0.5 + place.uniform(-0.2, 0.2, 3)
    i = np.arange(side) + 0.5 - side / 2
    dz, dx = (v.reshape(-1) * 0.5 for v in np.meshgrid(i, i, indexing="ij"))
    n = side * side
    iso = centre + np.stack([dx, np.zeros(n), dz], 1) @ M.T
    # the pixel pitch shrinks with the beamlet's obliqueness, alike for beamlets equally far out
    bs = (0.125 / np.sqrt(1.0 + (dx ** 2 + dz ** 2) / SAD ** 2)).astype(np.float32)
    src = (iso + M @ np.array([0.0, -SAD, 0.0])).astype(np.float32)
    # depth range: corner rays and axis of the 16-pixel field against the faces of the box
    near, far = np.full(n, np.inf), np.full(n, -np.inf)
    hi = np.array(dims) * VOXEL
    h = 8.0 * bs.astype(np.float64)
    for sx, sz in ((1, 1), (1, -1), (-1, 1), (-1, -1), (0, 0)):
        d = np.stack([sx * h, np.full(n, SAD), sz * h], 1) @ M.T
        for j in range(3):
            for face in (0.0, hi[j]):
                alpha = (face - src[:, j]) / d[:, j]
                p = src + d * alpha[:, None]
                o = [k for k in range(3) if k != j]
                ok = ((p[:, o] >= 0) & (p[:, o] <= hi[o])).all(1)
                near = np.where(ok, np.minimum(near, alpha * SAD), near)
                far = np.where(ok, np.maximum(far, alpha * SAD), far)
    near, far = near.astype(np.float32), far.astype(np.float32)
    L = np.ceil((far - near) / np.float32(VOXEL)).astype(np.int64)
    flu = np.zeros((n, 16, 16), np.float32)
    flu[:, 6:10, 6:10] = rng.uniform(0.8, 1.2, (n, 1, 1))
    return dict(n=n, dims=dims, angles=angles, M=M, iso=iso.astype(np.float32), bs=bs, src=src, near=near, far=far, L=L,
                Lmax=int(L.max()), flu=flu.reshape(n, NPIX), density=_slab_density(dims, case["medium"], rng),
                spectrum=_spectrum(rng), kernel=_kernel(rng, case["phi"]))


def _bev_inputs(p, seed):
    """Terma, mean density and dose on the BEV grids (n, Lmax, 256) of beamlets that have not been through
    the earlier stages: a beam attenuated in a layered medium, lit in its 4 x 4 open pixels."""
    g, dev = _generator(seed + 1), _device()
    n, Lm = p["n"], p["Lmax"]
    layers = torch.rand((n, Lm // 8 + 2), generator=g, device=dev).repeat_interleave(8, 1)[:, :Lm]
    rho = (0.2 + 1.6 * layers)[:, :, None] * (0.97 + 0.06 * torch.rand((n, Lm, NPIX), generator=g, device=dev))
    inside = torch.arange(Lm, device=dev)[None, :, None] < torch.as_tensor(p["L"], device=dev)[:, None, None]
    rho = torch.where(inside, rho, 0.0)
    depth = torch.exp(-0.05 * VOXEL * rho.mean(2, keepdim=True).cumsum(1))
    terma = torch.as_tensor(p["flu"], device=dev)[:, None, :] * depth * 0.06
    r = torch.arange(16, device=dev) - 7.5
    lateral = torch.exp(-(r[:, None] ** 2 + r[None, :] ** 2) / 18.0).reshape(1, 1, NPIX) + 2e-3
    dose = depth * lateral * (0.9 + 0.2 * torch.rand((n, Lm, NPIX), generator=g, device=dev))
    return [torch.where(inside, v, 0.0).float().contiguous() for v in (terma, rho, dose)]


def _beam_array(p):
    beams = (fd.Beam * p["n"])()
    for i, b in enumerate(beams):
        for j in range(3):
            b.isocenter[j], b.angles[j], b.source[j] = p["iso"][i, j], p["angles"][j], p["src"][i, j]
        b.beamlet_size[0] = b.beamlet_size[1] = p["bs"][i]
        b.fmap_size[0] = b.fmap_size[1] = 16
        b.sad, b.long_spacing = SAD, VOXEL
        b.lim_min, b.lim_max, b.long_dim = p["near"][i], p["far"][i], int(p["L"][i])
    return beams


def _context(dims, density, spectrum=None, kernel=None, seed=0, options=0):
    s, k = synth.synthetic_spectrum(seed), synth.synthetic_kernel(seed)
    if spectrum is not None:
        for i in range(12):
            s.energy[i], s.fluence[i], s.mu[i] = (v[i] for v in spectrum)
    if kernel is not None:
        k.n_phi = len(kernel["phi"])
        for i in range(8):
            k.theta_begin[i], k.theta_end[i], k.theta_mid[i] = (kernel[f][i] for f in ("begin", "end", "mid"))
            k.A[i], k.a[i], k.B[i], k.b[i] = (kernel[f][i] for f in "AaBb")
        for i, v in enumerate(kernel["phi"]):
            k.phi[i] = v
    return fd.Context(synth.make_volume(dims, VOXEL), density, s, k, options=options)


def _body(dims, seed):
    """A body of smooth random density (0.2-1.8 g/cc) in air, and an ellipsoidal target in four segments."""
    X, Y, Z = dims
    g, dev = _generator(seed + 2), _device()
    coarse = torch.rand((1, 1, Z // 6, Y // 6, X // 6), generator=g, device=dev)
    rho = 0.2 + 1.6 * torch.nn.functional.interpolate(coarse, size=(Z, Y, X), mode="trilinear")[0, 0]
    z, y, x = (torch.arange(d, device=dev, dtype=torch.float32) + 0.5 for d in (Z, Y, X))
    u, v, w = x[None, None, :] - X / 2, y[None, :, None] - Y / 2, z[:, None, None] - Z / 2
    inside = (u / (0.45 * X)) ** 2 + (v / (0.40 * Y)) ** 2 + (w / (0.47 * Z)) ** 2 <= 1.0
    rho = torch.where(inside, rho, 0.0012).contiguous()
    target = (u / (0.11 * X)) ** 2 + (v / (0.075 * Y)) ** 2 + (w / (0.08 * Z)) ** 2 <= 1.0
    edge = [X / 2 + 0.11 * X * f for f in (-1.1, -0.5, 0.0, 0.5, 1.1)]
    segments = [(target & (x >= a) & (x < b)[None, None, :]).to(torch.uint8).contiguous()
                for a, b in zip(edge, edge[1:])]
    isos = []
    for m in segments:
        at = m.nonzero().double().mean(0).cpu().numpy()[::-1]
        isos.append(((at + 0.5) * VOXEL).astype(np.float32))
    return rho.cpu().numpy(), segments, isos


def _bundles(case, isos, rng):
    """Beams of a 4pi plan, evenly over the sphere, dealt to the target's segments in turn."""
    n = case["beams"]
    start, of = int(rng.integers(180)), []
    for i, j in enumerate((start + np.arange(n) * max(1, 180 // n)) % 180):
        gantry, couch = synth.direction_to_varian_iec(synth.fibonacci_sphere(180)[j])
        deg = (round(math.degrees(gantry), 4), round(math.degrees(couch) + float(rng.uniform(-1, 1)), 4), 0.0)
        of.append((i % 4, synth.make_bundle(isos[i % 4], deg, fluence_dim=case["fluence"])))
    return of


def _plan(case, seed):
    dims = _dims(case)
    density, segments, isos = _body(dims, seed)
    ctx = _context(dims, density, seed=seed)
    bundles = _bundles(case, isos, _place(case))
    per = []
    for s, b in bundles:
        flags = ctx.beamlet_flags(segments[s], [b])[0]
        per.append(host.beamlets_init(b, flags, ctx.vol))
    return ctx, per


def _joined(per):
    """Beamlets, fluence and per-beam counts of several beams, as the batched calls take them."""
    counts = np.array([len(b) for b, _ in per], np.int32)
    beams, o = (fd.Beam * int(counts.sum()))(), 0
    for b, _ in per:
        ctypes.memmove(ctypes.byref(beams, o), b, ctypes.sizeof(b))
        o += ctypes.sizeof(b)
    return beams, np.concatenate([f for _, f in per], 0), counts


def _pencil_matrix(case, seed):
    """A dose matrix in CSR form on the device: beams of parallel pencils through the volume's middle,
    patch x patch voxels of each slice across the beam's main axis."""
    X, Y, Z = _dims(case)
    g, dev = _generator(seed + 4), _device()
    rng = _place(case)
    n, h = case["rows"], case["patch"]
    stride = np.array([1, X, X * Y])
    counts, columns, values = [], [], []
    for j in range(case["beams"]):
        d = synth.fibonacci_sphere(180)[int(rng.integers(180))]
        a = int(np.argmax(np.abs(d)))
        o = [k for k in range(3) if k != a]
        N = (X, Y, Z)[a]
        t = torch.arange(N, device=dev, dtype=torch.float32) + 0.5 - N / 2
        spread = 0.22 * torch.rand((2, n, 1), generator=g, device=dev) - 0.11
        col = (torch.arange(N, device=dev) * int(stride[a]))[None, :, None, None]
        ok = torch.ones((1, 1, 1, 1), dtype=torch.bool, device=dev)
        for q, k in enumerate(o):
            D = (X, Y, Z)[k]
            at = (D / 2 + spread[q] * D + t[None, :] * float(d[k] / d[a]) - h / 2).floor().long()
            at = at[:, :, None, None] + torch.arange(h, device=dev).reshape((1, 1, h, 1) if q else (1, 1, 1, h))
            ok = ok & (at >= 0) & (at < D)
            col = col + at * int(stride[k])
        col = torch.where(ok, col, X * Y * Z).expand(n, N, h, h).reshape(n, -1).sort(1).values
        real = col < X * Y * Z
        r = torch.arange(h, device=dev) - (h - 1) / 2
        counts.append(real.sum(1))
        columns.append(col[real])
        w = torch.rand((int(columns[-1].numel()),), generator=g, device=dev)
        values.append(0.01 + 0.99 * w ** 4)  # a few large entries, a broad tail
    return torch.cat(counts), torch.cat(columns), torch.cat(values)


def prepare(case, seed):
    kind = case["kind"]
    if kind in STAGES:
        p = _pencils(case, seed)
        options = (fd.FD_OPT_EXACT_G if case.get("exact_g") else 0) | (fd.FD_OPT_RPL_FP64_ALL if case.get("rpl64") else 0)
        s = dict(kind=kind, ctx=_context(p["dims"], p["density"], p["spectrum"], p["kernel"], options=options),
                 beams=_beam_array(p), stride=p["Lmax"] * NPIX, flu=torch.as_tensor(p["flu"], device=_device()))
        zero = torch.zeros(p["n"] * p["Lmax"] * NPIX, device=_device())
        s["terma"], s["density"], s["dose"] = zero, zero.clone(), zero.clone()
        if kind in ("cccs", "resample"):
            bev = [v.reshape(-1) for v in _bev_inputs(p, seed)]
            s["terma"], s["density"] = bev[:2]
            if kind == "resample":
                s["dose"] = bev[2]
        return s
    if kind in ("matrix", "plan", "serve"):
        ctx, per = _plan(case, seed)
        s = dict(kind=kind, ctx=ctx, cols=case["x"] * case["y"] * case["z"])
        if kind == "matrix":
            s["beams"], s["flu"] = per[0]
            return s
        s["type"] = VALUE_TYPES[case["type"]]
        s["batch"] = _joined(per)
        s["x"] = torch.rand((len(s["batch"][0]), case["k"]), generator=_generator(seed + 6), device=_device())
        if kind == "serve":
            rng, k, s["requests"] = np.random.default_rng(seed + 7), 0, []
            while k < len(per):
                take = int(rng.integers(1, 5))
                s["requests"].append(_joined(per[k:k + take]))
                k += take
            s["server"] = fd.Server(ctx)
        return s
    if kind == "product":
        counts, columns, values = _pencil_matrix(case, seed)
        offsets = torch.cat([counts.new_zeros(1), counts.cumsum(0)])
        dm = fd.DoseMat(case["x"] * case["y"] * case["z"])
        csr = fd.CSR(len(counts), len(columns), len(columns), offsets.data_ptr(), columns.data_ptr(), values.data_ptr())
        torch.cuda.synchronize()
        _lib.call("fd_dosemat_add_csr", dm._h, ctypes.byref(csr), None)
        op = fd.Spmm(dm, VALUE_TYPES[case["type"]])
        x = torch.rand((len(counts), case["k"]), generator=_generator(seed + 6), device=_device())
        return dict(kind=kind, op=op, x=x)
    if kind == "dense":
        return dict(kind=kind, dense=_dense(case, seed))
    density, segments, isos = _body(_dims(case), seed)
    mask = sum(segments).to(torch.uint8).contiguous()
    return dict(kind=kind, ctx=_context(_dims(case), density, seed=seed), mask=mask,
                bundles=[b for _, b in _bundles(case, isos, np.random.default_rng(seed + 3))])


def _dense(case, seed):
    """Rows whose nonzeros come in runs of about ten, as a beamlet's voxels do along x."""
    g, dev = _generator(seed + 8), _device()
    rows, cols = case["rows"], case["cols"]
    runs = rows * (cols // 10)
    on = torch.zeros((runs,), dtype=torch.bool, device=dev)
    on[torch.randperm(runs, generator=g, device=dev)[:max(1, round(case["fill"] * runs))]] = True
    v = torch.rand((rows, cols), generator=g, device=dev) + 1e-3
    v[:, :cols // 10 * 10] *= on.reshape(rows, -1).repeat_interleave(10, 1)
    v[:, cols // 10 * 10:] = 0.0
    return v


# ------------------------------------------------------------------ the calls


def run(state):
    kind = state["kind"]
    if kind in STAGES:
        ctx, beams, stride = state["ctx"], state["beams"], state["stride"]
        out = {}
        if kind in ("stages", "terma"):
            ctx.terma(beams, state["flu"], state["terma"], state["density"], stride)
            out.update(terma=state["terma"], density=state["density"])
        if kind in ("stages", "cccs"):
            ctx.cccs(beams, state["terma"], state["density"], state["dose"], stride)
            out.update(dose=state["dose"])
        if kind in ("stages", "resample"):
            out["offsets"], out["columns"], out["values"] = ctx.resample_csr(beams, state["dose"], stride)
        return out
    if kind == "matrix":
        dm = fd.DoseMat(state["cols"])
        dm.add_beam(state["ctx"], state["beams"], state["flu"])
        offsets, columns, values = dm.matrix(0)
        return dict(offsets=offsets, columns=columns, values=values)
    if kind in ("plan", "serve"):
        dm = fd.DoseMat(state["cols"])
        if kind == "plan":
            dm.add_beams(state["ctx"], *state["batch"])
        else:
            ids = [state["server"].submit(*r) for r in state["requests"]]
            for i in ids:
                state["server"].fetch(i, dm)
        with fd.Spmm(dm, state["type"]) as op:
            return dict(dose=op.run(state["x"]))
    if kind == "product":
        return dict(dose=state["op"].run(state["x"]))
    if kind == "dense":
        offsets, columns, values = host.dense_to_csr(state["dense"])
        return dict(offsets=offsets, columns=columns, values=values)
    return dict(flags=np.concatenate(state["ctx"].beamlet_flags(state["mask"], state["bundles"])))


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    kind = case["kind"]
    b = f = 0.0
    if kind in ("product", "dense", "flags"):
        if kind == "dense":
            cells = case["rows"] * case["cols"]
            return dict(bytes=4.0 * cells + 12.0 * case["fill"] * cells, flops=0.0)
        voxels = case["x"] * case["y"] * case["z"]
        if kind == "flags":
            return dict(bytes=float(voxels + case["beams"] * case["fluence"] ** 2),
                        flops=30.0 * 9 * case["beams"] * case["fluence"] ** 2 * 1.2 * case["x"] / 2)
        rows = case["beams"] * case["rows"]
        nnz = rows * case["patch"] ** 2 * (voxels ** (1 / 3))
        k = case["k"]
        return dict(bytes=nnz * (4 + (4 if case["type"] == "f32" else 2)) + 4.0 * k * (rows + voxels),
                    flops=2.0 * nnz * k)
    voxels = case["x"] * case["y"] * case["z"]
    if kind in STAGES:
        n, L = case["side"] ** 2, 1.2 * case["y"]
        steps, stages = ("terma", "cccs", "resample") if kind == "stages" else (kind,), ()
    else:
        n, L = 133 * case["beams"], 1.15 * case["x"]
        steps = ("terma", "cccs", "resample")
    bev, nnz = n * L * NPIX, n * L * 80.0
    phi = case.get("phi", 8)
    if "terma" in steps:
        b += 4.0 * (n * NPIX + voxels + 2 * bev)
        f += bev * 4 * 25
    if "cccs" in steps:
        b += 4.0 * bev * (3 if kind == "cccs" else 1)
        f += 40.0 * 47.7e3 * L * n * phi / 8
    if "resample" in steps:
        b += 12.0 * nnz + (4.0 * bev if kind == "resample" else 0.0)
        f += nnz * 125 * 30
    if kind in ("plan", "serve"):  # the operator is written once, read once, and the dose written
        b += nnz * 2 * (4 + (4 if case["type"] == "f32" else 2)) + 4.0 * case["k"] * (voxels + n)
        f += 2.0 * nnz * case["k"]
    return dict(bytes=b, flops=f)


# ------------------------------------------------------------------ the same in 64 bits


def exact(case, seed):
    kind = case["kind"]
    if kind in STAGES:
        p = _pencils(case, seed)
        if p["n"] * p["Lmax"] > 80_000 or case["phi"] > 8 and p["n"] > 64:
            return None
        out = {}
        terma, rho, dose = _bev_inputs(p, seed) if kind in ("cccs", "resample") else (None, None, None)
        if kind in ("stages", "terma"):
            terma, rho = _terma64(p)
            out.update(terma=terma.reshape(-1), density=rho.reshape(-1))
        if kind in ("stages", "cccs"):
            dose = _cccs64(p, terma.double(), rho.double(), bool(case.get("exact_g")))
            out.update(dose=dose.reshape(-1))
        if kind in ("stages", "resample"):
            out.update(offsets=None, columns=None, values=_resample64(p, dose))
        return out
    if kind == "product":
        counts, columns, values = _pencil_matrix(case, seed)
        k = case["k"]
        x = torch.rand((len(counts), k), generator=_generator(seed + 6), device=_device()).double()
        row = torch.repeat_interleave(torch.arange(len(counts), device=x.device), counts)
        y = torch.zeros((case["x"] * case["y"] * case["z"], k), dtype=torch.float64, device=x.device)
        part = max(1, (1 << 27) // k)
        for i in range(0, len(columns), part):
            e = slice(i, i + part)
            y.index_add_(0, columns[e], values[e].double()[:, None] * x[row[e]])
        return dict(dose=y)
    if kind == "dense":
        dense = _dense(case, seed)
        return dict(offsets=None, columns=None, values=dense[dense != 0].double())
    return None  # whole plans take a CPU minutes in 64 bits; flags are whole numbers


def _fma(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _terma64(p):
    """Terma and mean density (n, Lmax, 256): four samples a slice along each pixel's ray, trilinear
    density (zero outside), the spectrum attenuated by the radiological path so far."""
    dev = _device()
    X, Y, Z = p["dims"]
    padded = torch.zeros((Z + 2, Y + 2, X + 2), dtype=torch.float64, device=dev)
    padded[1:-1, 1:-1, 1:-1] = torch.as_tensor(p["density"], device=dev)
    flat = padded.reshape(-1)
    energy, weight, mu = (torch.as_tensor(v, device=dev).double() for v in p["spectrum"])
    M = torch.as_tensor(p["M"], device=dev)
    r = torch.arange(16, device=dev).double() - 7.5
    terma = torch.zeros((p["n"], p["Lmax"], NPIX), dtype=torch.float64, device=dev)
    rho_out = torch.zeros_like(terma)
    for i in range(p["n"]):
        L, bs = int(p["L"][i]), float(p["bs"][i])
        ray = torch.stack([(r * bs).repeat(16), torch.full((NPIX,), SAD, dtype=torch.float64, device=dev),
                           (r * bs).repeat_interleave(16)], 1) @ M.T
        dt = VOXEL / (4 * SAD)
        t = float(p["near"][i]) / SAD + dt * (torch.arange(4 * L, device=dev).double() + 1)
        pos = (torch.as_tensor(p["src"][i], device=dev).double() + ray[None] * t[:, None, None]) / VOXEL - 0.5
        cell = pos.floor()
        w = pos - cell
        cell = cell.long()
        rho = torch.zeros((4 * L, NPIX), dtype=torch.float64, device=dev)
        for c in range(8):
            o = [(c >> j) & 1 for j in range(3)]
            q = [(cell[..., j] + o[j] + 1).clamp(0, d + 1) for j, d in enumerate((X, Y, Z))]
            part = flat[(q[2] * (Y + 2) + q[1]) * (X + 2) + q[0]]
            for j in range(3):
                part = part * (w[..., j] if o[j] else 1 - w[..., j])
            rho += part
        path = (rho * (ray.norm(dim=1) * dt)).cumsum(0)
        att = sum(weight[e] * energy[e] * mu[e] * torch.exp(-mu[e] * path) for e in range(12))
        att = att / (t * t)[:, None] * torch.as_tensor(p["flu"][i], device=dev).double()
        terma[i, :L] = att.reshape(L, 4, NPIX).mean(1)
        rho_out[i, :L] = rho.reshape(L, 4, NPIX).mean(1)
    return terma, rho_out


def _cccs64(p, terma, rho, exact_g):
    """Collapsed-cone recursion along the rays of every forward cone and azimuth.  The 256 rays of an
    azimuth share one march through the lattice (in FP32, as the march defines the voxels crossed); the
    recursion on them is in 64 bits."""
    dev, n, K = _device(), p["n"], p["kernel"]
    L = torch.as_tensor(p["L"], device=dev)
    bs = torch.as_tensor(p["bs"], device=dev)[:, None]
    near = torch.as_tensor(p["near"], device=dev).double()[:, None, None]
    P = len(K["phi"])
    ix, iy = torch.arange(NPIX, device=dev) % 16, torch.arange(NPIX, device=dev) // 16
    dose = torch.zeros_like(terma)
    rows = torch.arange(n, device=dev)
    eps, far_eps = float(np.float32(1e-4)), torch.tensor(np.float32(1e-3), device=dev)

    def step(c, d):
        up = (c + far_eps).ceil() - c
        down = (c - far_eps).floor() - c
        return torch.where(d > 0, up * (1 / d), torch.where(d < 0, down * (1 / d), torch.inf))

    def mean_kernel(x):
        return torch.where(x < 1e-4, 1 - x / 2 + x * x / 6, -torch.expm1(-x) / x.clamp(min=1e-30)) if exact_g else 1.0

    for t in range(8):
        th = float(K["mid"][t])
        if th > math.pi / 2:
            continue
        A, a, B, b = (float(K[f][t]) for f in "AaBb")
        ph = torch.as_tensor(K["phi"], device=dev).double()
        u = [(math.sin(th) * ph.cos()).float(), (math.sin(th) * ph.sin()).float(),
             torch.full((P,), math.cos(th), dtype=torch.float64, device=dev).float()]
        v = [u[0] / bs, u[1] / bs, (u[2] / VOXEL).expand(n, P)]
        norm = 1 / (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]).sqrt()
        d = [c * norm for c in v]
        at = [torch.full((n, P), c, device=dev) for c in (0.5, 0.5, 0.0)]
        XA = torch.zeros((n, P, NPIX), dtype=torch.float64, device=dev)
        XB = torch.zeros_like(XA)
        s = torch.zeros(n, dtype=torch.long, device=dev)
        while bool((s < L).any()):
            z = s.clamp(max=terma.shape[1] - 1)
            Ts, Rs = (w[rows, z][:, None, :].expand(n, P, NPIX) for w in (terma, rho))
            D, C = (torch.zeros((n, NPIX), dtype=torch.float64, device=dev) for _ in range(2))
            live = (s < L)[:, None].expand(n, P)
            while bool(live.any()):
                sz = step(at[2], d[2])
                go = torch.minimum(torch.minimum(step(at[0], d[0]), step(at[1], d[1])), sz)
                to = [_fma(go, e, c) for e, c in zip(d, at)]
                end = (to[2] - to[2].round()).abs() < eps
                snap = [_fma(sz, e, c) for e, c in zip(d, at)]
                snap[2] = snap[2].round()
                to = [torch.where(end, q, w) for q, w in zip(snap, to)]
                mx, my = ((q + w)[..., None].mul(0.5).floor().long() for q, w in zip(at[:2], to[:2]))
                m = (mx + ix) % 16 + 16 * ((my + iy) % 16)
                # physical distance of the ray's two lattice points, the lateral pitch growing with depth
                ends = []
                for c in (at, to):
                    depth = c[2].double()[..., None] * VOXEL
                    grow = (depth + near) / SAD * bs.double()[..., None]
                    ends.append(((c[0].double()[..., None] + ix - 8) * grow,
                                 (c[1].double()[..., None] + iy - 8) * grow, depth))
                T, R = Ts.gather(2, m), Rs.gather(2, m)
                q = sum((e1 - e0) ** 2 for e0, e1 in zip(*ends)).sqrt() * R
                ga, gb = mean_kernel(a * q), mean_kernel(b * q)
                part = (A / a * ((1 - ga) * T + ga * XA) + B / b * ((1 - gb) * T + gb * XB)) * q
                on = live[..., None]
                D.scatter_add_(1, m.reshape(n, -1), torch.where(on, part, 0.0).reshape(n, -1))
                C.scatter_add_(1, m[:, -1], torch.where(on, q, 0.0)[:, -1])
                cross = torch.zeros_like(m, dtype=torch.bool)
                for c0, c1, i in ((at[0], to[0], ix), (at[1], to[1], iy)):
                    f0, f1 = (c.floor().long()[..., None] + i for c in (c0, c1))
                    cross |= f0.div(16, rounding_mode="floor") != f1.div(16, rounding_mode="floor")
                for X, c in ((XA, a), (XB, b)):
                    e = torch.exp(-c * q)
                    new = torch.where(cross, 0.0, T * (1 - e) + e * X)
                    X.copy_(torch.where(on, new, X))
                at = [torch.where(live, w, c) for w, c in zip(to, at)]
                live = live & ~end
            out = D / (C + eps)
            dose[rows, z] += torch.where((s < L)[:, None], out, 0.0)
            s = torch.where(s < L, torch.maximum(at[2][:, 0].round().long(), s + 1), s)
    return dose


def _resample64(p, dose, extent=2.0):
    """Nonzero voxel values of every beamlet, in voxel order: the mean of the BEV dose under 5^3 points of
    each voxel near the beamlet's axis.  Which BEV cell a point falls in is decided in FP32."""
    dev = _device()
    X, Y, Z = p["dims"]
    f32 = dict(dtype=torch.float32, device=dev)
    N = torch.as_tensor(np.ascontiguousarray(p["M"].T).astype(np.float32), device=dev)

    def bev(q, src):
        c = [w - o for w, o in zip(q, src)]
        return [_fma(N[r, 2], c[2], _fma(N[r, 1], c[1], N[r, 0] * c[0])) for r in range(3)]

    vs = torch.tensor(VOXEL, **f32)
    half = (vs * vs + vs * vs + vs * vs).sqrt() * 0.5
    z, y, x = torch.meshgrid(*(torch.arange(k, device=dev) for k in (Z, Y, X)), indexing="ij")
    x, y, z = (w.reshape(-1) for w in (x, y, z))
    o = (torch.arange(5, **f32) + 0.5) * np.float32(1 / np.float32(5))
    ok_, oj, oi = (w.reshape(-1) for w in torch.meshgrid(o, o, o, indexing="ij"))
    found = []
    for i in range(p["n"]):
        src = [torch.tensor(float(c), **f32) for c in p["src"][i]]
        c = bev([(w + 0.5) * vs for w in (x, y, z)], src)
        near_axis = (c[0] * c[0] + c[2] * c[2]).sqrt() <= half + extent
        big = bev([(8 * vs) * (w.div(8, rounding_mode="floor") + 0.5) for w in (x, y, z)], src)
        near_axis &= (big[0] * big[0] + big[2] * big[2]).sqrt() < extent + 8 * half
        sel = near_axis.nonzero()[:, 0]
        q = [(w[sel].float()[:, None] + off) * vs for w, off in ((x, oi), (y, oj), (z, ok_))]
        c = bev(q, src)
        k = torch.tensor(SAD, **f32) / torch.tensor(float(p["bs"][i]), **f32)
        dd = (c[1] - torch.tensor(float(p["near"][i]), **f32)) * (1 / vs)
        inv = 1 / c[1]
        u, w = _fma(c[0] * k, inv, torch.tensor(8.0, **f32)), _fma(c[2] * k, inv, torch.tensor(8.0, **f32))
        inside = (dd >= 0) & (dd < int(p["L"][i])) & (u >= 0) & (u < 16) & (w >= 0) & (w < 16)
        cell = dd.long().clamp(0, dose.shape[1] - 1) * NPIX + w.long().clamp(0, 15) * 16 + u.long().clamp(0, 15)
        v = torch.where(inside, dose[i].reshape(-1).double()[cell], 0.0).sum(1) / 125
        found.append(v[v != 0])
    return torch.cat(found)
