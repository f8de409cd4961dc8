"""Performance cases of the reconstruction core: what a user has it do, through its public entry points.

Kinds (`case["kind"]`), each with the sizes it is run at:

  operators   one tilt through the operator calls of a host loop (fp_march, compare, crop_border, bp)
  sart        one iteration of the SART driver from an empty volume (fp32 or half volume)
  sart_ctf    the same with 3D-CTF defocus slabs
  subvol      one pass of a batched sub-volume WBP plan over cubes of 32 .. 128 voxels, with or without CTF
  prep        projection preparation of a stack, for SART (band-pass, dose weighting) or WBP (ramp)
  pair_grad   one training step over (sub-volume, tilt) pairs: projections, loss, gradients of the
              sub-volumes and the shifts
  pair_search the integer shift search over the same pairs
  project     one training step of a whole volume through a tilt series, gradients of volume and shifts

Measured projections are Gaussian densities projected in closed form plus noise; they come from the
seed and torch alone, so every build of the library sees the same inputs.  `exact` evaluates a case in
float64 with torch operations: every ray sample, every voxel's sub-rays, every FFT.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import artiatomi_amd as A
from artiatomi_amd import autograd as AG

F64 = torch.float64


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest calls: one tilt of a small sub-tomogram, operator by operator, as a host program
        # that keeps its own loop drives the library; launches and call overhead count
        dict(name="operators_64", kind="operators", nx=64, ny=64, nz=32, width=72, height=60, tilt=27.0, os=1),
        # a coarse (binned) tomogram: the repository's small SART workload, no tilt-axis rotation
        dict(name="sart_256", kind="sart", nx=256, ny=256, nz=64, width=256, height=256, tilts=41, step=3.0, os=1,
             sirt=1, psi=0.0, shift=0.0, half=False),
        # the repository's full-size SART workload: rotated tilt axis, shifts, two-fold oversampling
        dict(name="sart_1024", kind="sart", nx=1024, ny=1024, nz=256, width=1024, height=1024, tilts=61, step=2.0,
             os=2, sirt=1, psi=5.0, shift=5.0, half=False),
        # ordered subsets over a half-precision volume of uneven size, detector larger than the volume
        dict(name="sart_half_ragged", kind="sart", nx=480, ny=372, nz=101, width=531, height=393, tilts=28, step=4.0,
             os=2, sirt=4, psi=4.0, shift=3.0, half=True),
        # SART with 3D-CTF correction of a binned tomogram
        dict(name="sart_ctf_512", kind="sart_ctf", nx=512, ny=512, nz=128, width=512, height=512, tilts=21, step=6.0,
             os=2, sirt=1, psi=0.0, shift=2.0, pixel_nm=0.5, slab_nm=8.0),
        # sub-volume WBP of particles picked from a tomogram: cubes in ratio 4:3:2:1, extra shifts
        dict(name="subvol_300", kind="subvol", cubes=300, field=2048, depth=512, width=2048, height=2048, tilts=41,
             step=3.0, os=2, ctf=False),
        # the same with 3D-CTF slabs at full detector size
        dict(name="subvol_ctf_4096", kind="subvol", cubes=400, field=4096, depth=1024, width=4096, height=4096,
             tilts=11, step=12.0, os=2, ctf=True),
        # preparing a full-size raw series for SART: 16-bit counts, band-pass, dose weighting
        dict(name="prep_4096", kind="prep", n=31, width=4096, height=4096, dtype="uint16", wbp=False),
        # preparing a binned series of uneven size for WBP (mirror padding, ramp)
        dict(name="prep_wbp_ragged", kind="prep", n=41, width=960, height=927, dtype="int16", wbp=True),
        # gradient-based refinement of particles: one step over all (particle, tilt) pairs
        dict(name="pair_grad_100", kind="pair_grad", cubes=100, n=64, field=512, depth=128, width=512, height=512,
             tilts=41, step=3.0, margin=8),
        # cross-correlation refinement of particles, shifts up to 12 pixels
        dict(name="pair_search_100", kind="pair_search", cubes=100, n=48, field=512, depth=128, width=512, height=512,
             tilts=41, step=3.0, margin=14, max_shift=12),
        # gradient of a whole tomogram and its per-tilt shifts
        dict(name="project_512", kind="project", nx=512, ny=512, nz=128, width=512, height=512, tilts=13, step=10.0,
             psi=0.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _quad(n):
    return max(4, n - n % 4)   # volumes are a multiple of 4 voxels wide


def draw(rng):
    kind = rng.choice(["operators", "sart", "sart", "sart_ctf", "subvol", "subvol", "prep", "prep", "pair_grad",
                       "pair_search", "project"])
    if kind == "operators":
        n = _log(rng, 32, 256)
        nx, ny = _quad(n), rng.randint(n // 2, n)
        return dict(kind=kind, nx=nx, ny=ny, nz=_log(rng, 16, 96), width=nx + rng.randint(-5, 20),
                    height=ny + rng.randint(-5, 20), tilt=rng.uniform(-60.0, 60.0), os=rng.choice([1, 2]))
    if kind in ("sart", "sart_ctf"):
        n = _log(rng, 96, 512) if kind == "sart" else _log(rng, 96, 384)
        nx, ny, nz = _quad(n), rng.randint(2 * n // 3, n), rng.randint(n // 6, n // 3)
        step = rng.choice([3.0, 4.0, 5.0, 6.0])
        c = dict(kind=kind, nx=nx, ny=ny, nz=nz, width=nx + rng.randint(-9, 40), height=ny + rng.randint(-9, 40),
                 tilts=rng.randint(5, 15), step=step, os=rng.choice([1, 2]), sirt=rng.choice([1, 1, 3]),
                 psi=rng.choice([0.0, 5.0]), shift=rng.choice([0.0, 4.0]))
        if kind == "sart":
            return dict(c, half=rng.random() < 0.3)
        return dict(c, pixel_nm=rng.choice([0.25, 0.5, 0.8]), slab_nm=rng.choice([4.0, 8.0, 16.0]))
    if kind == "subvol":
        field = rng.choice([512, 1000, 1024, 2048])
        return dict(kind=kind, cubes=_log(rng, 10, 150), field=field, depth=field // 4,
                    width=field - rng.choice([0, 0, 12, 74]), height=field - rng.choice([0, 0, 12, 74]),
                    tilts=rng.randint(5, 15), step=8.0, os=rng.choice([1, 2]), ctf=rng.random() < 0.5)
    if kind == "prep":
        n = rng.choice([256, 512, 960, 1000, 1024, 1920, 2048, rng.randint(200, 2000)])
        return dict(kind=kind, n=rng.randint(3, 24), width=n, height=n - rng.choice([0, 0, 33, n // 12]),
                    dtype=rng.choice(["int16", "uint16", "float32"]), wbp=rng.random() < 0.5)
    if kind == "project":
        n = _log(rng, 64, 256)
        return dict(kind=kind, nx=_quad(n), ny=n, nz=rng.randint(n // 6, n // 3), width=n + rng.randint(-7, 30),
                    height=n + rng.randint(-7, 30), tilts=rng.randint(3, 13), step=10.0, psi=rng.choice([0.0, 5.0]))
    n = rng.choice([24, 32, 40, 48, 64])
    c = dict(kind=kind, cubes=_log(rng, 4, 60), n=n, field=512, depth=128, width=512, height=512,
             tilts=rng.randint(7, 31), step=4.0)
    if kind == "pair_grad":
        return dict(c, margin=rng.randint(4, 10))
    m = rng.randint(3, 16)
    return dict(c, margin=m + 2, max_shift=m)


# ------------------------------------------------------------------ inputs (seed and torch alone)

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _tilt_angles(case):
    n = case["tilts"]
    return [(i - (n - 1) / 2.0) * case["step"] for i in range(n)]


def _detector_point(tg, p):
    """Detector coordinates (pixels) of world points p (n, 3)."""
    M = np.array(list(tg.det_matrix), np.float64).reshape(4, 4)
    q = p @ M[:2, :3].T + M[:2, 3]
    return q[:, 0], q[:, 1]


class _Densities:
    """Isotropic Gaussian densities in a box and their projections in closed form."""

    def __init__(self, lo, hi, count, rng, sigma):
        self.c = rng.uniform(lo, hi, (count, 3))
        self.s = rng.uniform(sigma[0], sigma[1], count)
        self.a = rng.uniform(0.1, 1.0, count)

    def project(self, tg, W, H, x0=0, y0=0, shift=(0.0, 0.0)):
        x, y = _detector_point(tg, self.c)
        t = lambda v: torch.as_tensor(v, device=_device(), dtype=torch.float32)[:, None]  # noqa: E731
        px = torch.arange(W, device=_device(), dtype=torch.float32)[None] + (x0 + 0.5)
        py = torch.arange(H, device=_device(), dtype=torch.float32)[None] + (y0 + 0.5)
        g = lambda p, c: torch.exp(-0.5 * ((p - t(c)) / t(self.s)) ** 2)  # noqa: E731
        return (g(py, y + shift[1]) * t(self.a * self.s * math.sqrt(2 * math.pi))).T.contiguous() @ g(px, x + shift[0])


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _density_volume(d, vg):
    """The densities sampled at the voxel centres, (nz, ny, nx) float32."""
    ax = [torch.arange(n, device=_device(), dtype=torch.float32) + (0.5 + vg.bbox_min[i])
          for i, n in enumerate((vg.nx, vg.ny, vg.nz))]
    g = [torch.exp(-0.5 * ((ax[i][None] - torch.as_tensor(d.c[:, i], device=_device(), dtype=torch.float32)[:, None])
                           / torch.as_tensor(d.s, device=_device(), dtype=torch.float32)[:, None]) ** 2) for i in range(3)]
    vol = torch.zeros((vg.nz, vg.ny, vg.nx), device=_device())
    for b in range(len(d.a)):
        vol += float(d.a[b]) * g[2][b][:, None, None] * g[1][b][None, :, None] * g[0][b][None, None, :]
    return vol


def _series(case, seed):
    """Volume placement, tilt geometry and noisy projections of a whole-volume case."""
    rng = np.random.default_rng([int(seed), 1])
    vg = A.volume_geometry(case["nx"], case["ny"], case["nz"])
    W, H = case["width"], case["height"]
    tilts = _tilt_angles(case) if "tilts" in case else [case["tilt"]]
    psi, shift = case.get("psi", 0.0), case.get("shift", 0.0)
    psis = rng.uniform(-psi, psi, len(tilts)) if psi else np.zeros(len(tilts))
    shifts = rng.uniform(-shift, shift, (len(tilts), 2)) if shift else np.zeros((len(tilts), 2))
    acq = A.Acquisition.build(vg, W, H, tilts, psis_deg=psis.tolist(), shifts=shifts.tolist())
    lo, hi = np.array(list(vg.bbox_min)), np.array(list(vg.bbox_max))
    small = min(case["nx"], case["ny"], case["nz"])
    d = _Densities(lo, hi, 60, rng, (2.0, max(3.0, 0.2 * small)))
    projs = torch.empty((len(tilts), H, W), device=_device())
    for t, g in enumerate(acq.geoms):
        projs[t] = d.project(g, W, H)
    projs += torch.randn(projs.shape, generator=_generator(seed), device=_device()) * (0.05 * float(projs.max()))
    return vg, acq, projs, d


def _defocus(case, acq, rng):
    return [A.TiltDefocus(float(d), float(d) + 200.0, float(a), float(t))
            for d, a, t in zip(rng.uniform(2000.0, 5000.0, len(acq)), rng.uniform(-90.0, 90.0, len(acq)), acq)]


def _sart_inputs(case, seed):
    vg, acq, projs, _ = _series(case, seed)
    sp = A.sart_params(lambda_=0.3, sirt_count=case["sirt"], oversampling=case["os"])
    s = dict(vg=vg, acq=acq, projs=projs, sp=sp)
    if case["kind"] == "sart_ctf":
        s["ctf"] = A.ctf_params(pixelsize_nm=case["pixel_nm"], slice_thickness_nm=case["slab_nm"], amp_contrast=0.07)
        s["defocus"] = _defocus(case, acq.tilts_deg, np.random.default_rng([int(seed), 2]))
    return s


def _subvol_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 3])
    W, H, F, D = case["width"], case["height"], case["field"], case["depth"]
    tilts = _tilt_angles(case)
    full = A.volume_geometry(F, F, D)
    counts = [case["cubes"] * r // 10 for r in (4, 3, 2, 1)]
    counts[0] += case["cubes"] - sum(counts)
    sizes = [n for n, c in zip((32, 64, 96, 128), counts) for _ in range(c)]
    rng.shuffle(sizes)
    vgs, geoms = [], []
    for n in sizes:
        pos = rng.uniform([n / 2] * 3, [F - n / 2, F - n / 2, D - n / 2]) + 1.0
        vgs.append(A.subvolume_geometry(n, 1.0, (1.0, 1.0, 1.0), full, pos.tolist()))
        extra = rng.uniform(-4.0, 4.0, (len(tilts), 2))
        geoms.append([A.subvolume_tilt_geometry(t, W, H, extra_shift=extra[i]) for i, t in enumerate(tilts)])
    base = [A.tilt_geometry(t, W, H) for t in tilts]
    d = _Densities(np.array(list(full.bbox_min)), np.array(list(full.bbox_max)), 80, rng, (3.0, 40.0))
    gen = _generator(seed)
    images = torch.empty((len(tilts), H, W), device=_device())
    ramp = torch.fft.fftfreq(H, device=_device()).abs()[:, None].float()
    for t, g in enumerate(base):   # ramp-filtered projections, as a WBP series arrives
        img = d.project(g, W, H)
        img += torch.randn((H, W), generator=gen, device=_device()) * (0.05 * float(img.max()))
        images[t] = torch.fft.irfft2(torch.fft.rfft2(img) * ramp, s=(H, W))
    s = dict(full=full, vgs=vgs, geoms=geoms, images=images, kw={})
    if case["ctf"]:
        s["kw"] = dict(ctf=A.ctf_params(pixelsize_nm=0.25, slice_thickness_nm=4.0, amp_contrast=0.07),
                       slab_ranges=[A.defocus_distances(full, g) for g in base], defocus=_defocus(case, tilts, rng))
    return s


_TORCH = {"int16": torch.int16, "uint16": torch.uint16, "float32": torch.float32}
_PREP = {"int16": "int16", "uint16": "uint16", "float32": "float32"}


def _prep_inputs(case, seed):
    n, W, H = case["n"], case["width"], case["height"]
    gen = _generator(seed)
    N = max(W, H)
    # counts with a gradient, noise and hot pixels
    base = 200.0 + 60.0 * torch.linspace(0, 1, W, device=_device())[None] * torch.linspace(
        1, 0.5, H, device=_device())[:, None]
    images = torch.empty((n, H, W), device=_device(), dtype=_TORCH[case["dtype"]])
    for i in range(n):
        f = base + 20.0 * torch.randn((H, W), generator=gen, device=_device())
        hot = torch.randint(0, H * W, (max(1, H * W // 50000),), generator=gen, device=_device())
        f.view(-1)[hot] = 9000.0
        f = f if case["dtype"] == "float32" else f.round().clamp(0, 30000).to(torch.int16)
        images[i] = f.view(torch.uint16) if case["dtype"] == "uint16" else f
    tilts = [(-60.0 + 120.0 * i / max(1, n - 1)) for i in range(n)]
    common = dict(dtype=_PREP[case["dtype"]], lp=0.39 * N, lps=0.1 * N)
    if case["wbp"]:
        pp = A.prep_params(**common, wbp=True, wbp_method="ramp", normalization="std")
    else:
        pp = A.prep_params(**common, dose_weighting=True, pixelsize_nm=0.25, normalization="mean")
    return dict(pp=pp, images=images, tilts=tilts, psis=[2.0 + 0.05 * i for i in range(n)],
                dose=[0.5 * (i + 1) for i in range(n)], common=common)


def _pair_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 4])
    n, K, W, H = case["n"], case["cubes"], case["width"], case["height"]
    full = A.volume_geometry(case["field"], case["field"], case["depth"])
    base = [A.tilt_geometry(t, W, H) for t in _tilt_angles(case)]
    vols = torch.empty((K, n, n, n), device=_device())
    subs, pairs, geoms, targets = [], [], [], []
    true = rng.uniform(-3.0, 3.0, (K, len(base), 2))
    for k in range(K):
        pos = rng.uniform([n / 2] * 3, [case["field"] - n / 2] * 2 + [case["depth"] - n / 2]) + 1.0
        vg = A.subvolume_geometry(n, 1.0, (1.0, 1.0, 1.0), full, pos.tolist())
        lo, hi = np.array(list(vg.bbox_min)), np.array(list(vg.bbox_max))
        d = _Densities(lo + 0.35 * n, hi - 0.35 * n, 4, rng, (0.05 * n, 0.08 * n))   # zero margins
        vols[k] = _density_volume(d, vg)
        subs.append((vg, k * n ** 3))
        centre = (0.5 * (lo + hi))[None]
        for t, g in enumerate(base):
            # the cube's footprint and a margin, in the detector, of one size for every cube
            a = math.radians(_tilt_angles(case)[t])
            w = math.ceil(n * (math.cos(a) + abs(math.sin(a)))) + 2 * case["margin"]
            h = n + 2 * case["margin"]
            cx, cy = _detector_point(g, centre)
            x0, y0 = (int(min(max(0.0, round(c - e / 2)), D - e)) for c, e, D in ((cx[0], w, W), (cy[0], h, H)))
            pairs.append((k, x0, y0, w, h))
            geoms.append(g)
            targets.append(d.project(g, w, h, x0, y0, true[k, t]).reshape(-1))
    targets = torch.cat(targets)
    targets += torch.randn(targets.shape, generator=_generator(seed), device=_device()) * (0.05 * float(targets.max()))
    return dict(vols=vols.reshape(-1), subs=subs, pairs=pairs, geoms=geoms, targets=targets)


def _project_inputs(case, seed):
    vg, acq, projs, d = _series(case, seed)
    rng = np.random.default_rng([int(seed), 5])
    s = torch.as_tensor(rng.uniform(-2.0, 2.0, (len(acq.geoms), 2)), device=_device(), dtype=torch.float32)
    return dict(vg=vg, acq=acq, target=projs, vol=_density_volume(d, vg), shifts=s)


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    kind = case["kind"]
    ctx = A.ArtiaContext(torch.cuda.current_device())
    if kind == "operators":
        vg, acq, projs, d = _series(case, seed)
        W, H = case["width"], case["height"]
        return dict(case=case, ctx=ctx, vg=vg, acq=acq, real=projs[0].contiguous(), vol=_density_volume(d, vg),
                    proj=torch.empty((H, W), device="cuda"), dist=torch.empty((H, W), device="cuda"),
                    update=torch.empty((vg.nz, vg.ny, vg.nx), device="cuda"))
    if kind in ("sart", "sart_ctf"):
        s = _sart_inputs(case, seed)
        vg = s["vg"]
        dt = torch.float16 if case.get("half") else torch.float32
        return dict(s, case=case, ctx=ctx, vol=torch.empty((vg.nz, vg.ny, vg.nx), device="cuda", dtype=dt))
    if kind == "subvol":
        s = _subvol_inputs(case, seed)
        sizes = [g.nx * g.ny * g.nz for g in s["vgs"]]
        flat = torch.zeros(sum(sizes), device="cuda")
        subs, off = [], 0
        for g, k in zip(s["vgs"], sizes):
            subs.append((g, flat[off:off + k]))
            off += k
        # a program that reconstructs many series keeps one tuning
        plan = A.SubvolPlan(ctx, subs, s["geoms"], s["images"], oversampling=case["os"],
                            tuning=A.SubvolTuning(0, 1, 2 if case["ctf"] else 1, 8), **s["kw"])
        return dict(case=case, ctx=ctx, plan=plan, flat=flat)
    if kind == "prep":
        s = _prep_inputs(case, seed)
        out = torch.empty(s["images"].shape, device="cuda", dtype=torch.float32)
        return dict(s, case=case, ctx=ctx, out=out)
    if kind in ("pair_grad", "pair_search"):
        s = _pair_inputs(case, seed)
        ps = A.PairSet(ctx, s["subs"], s["pairs"], s["geoms"])
        shifts = torch.zeros((ps.npairs, 2), device="cuda")
        return dict(case=case, ctx=ctx, ps=ps, vols=s["vols"], targets=s["targets"], shifts=shifts)
    if kind == "project":
        s = _project_inputs(case, seed)
        acq = s["acq"]
        setup = AG.ProjectionSetup(ctx=ctx, vg=s["vg"], width=case["width"], height=case["height"],
                                   tilts_deg=acq.tilts_deg, psis_deg=acq.psis_deg)
        return dict(case=case, ctx=ctx, setup=setup, vol=s["vol"], shifts=s["shifts"], target=s["target"])
    raise ValueError(f"unknown kind {kind!r}")


def run(s):
    case = s["case"]
    kind, ctx = case["kind"], s["ctx"]
    if kind == "operators":
        vg, acq = s["vg"], s["acq"]
        proj, dist, upd = s["proj"].zero_(), s["dist"], s["update"].zero_()
        ctx.fp_march(vg, acq.geoms[0], s["vol"], proj, dist)
        ctx.compare(s["real"], proj, dist, acq.real_lengths[0])
        ctx.crop_border(proj, acq.hitpoints[0])
        ctx.bp(vg, acq.geoms[0], upd, proj, 0.3, oversampling=case["os"])
        return dict(residual=proj, dist=dist, update=upd)
    if kind == "sart":
        s["vol"].zero_()
        ctx.sart_run(s["vg"], s["acq"], s["projs"], s["vol"], s["sp"], iterations=1)
        return dict(volume=s["vol"])
    if kind == "sart_ctf":
        s["vol"].zero_()
        ctx.sart_ctf_run(s["vg"], s["acq"], s["defocus"], s["projs"], s["vol"], s["sp"], s["ctf"], iterations=1)
        return dict(volume=s["vol"])
    if kind == "subvol":
        s["flat"].zero_()
        s["plan"].execute()
        return dict(cubes=s["flat"])
    if kind == "prep":
        mean, std, bad = ctx.prepare_projections(s["pp"], s["images"], s["out"], tilt_deg=s["tilts"],
                                                 psi_deg=s["psis"], dose=s["dose"])
        return dict(out=s["out"], mean=mean, std=std, bad=bad)
    if kind == "pair_grad":
        vols, shifts = s["vols"].requires_grad_(True), s["shifts"].requires_grad_(True)
        vols.grad = shifts.grad = None
        images = AG.project_pairs(vols, shifts, s["ps"])
        (images - s["targets"]).square().sum().backward()
        return dict(images=images, grad_volumes=vols.grad, grad_shifts=shifts.grad)
    if kind == "pair_search":
        with torch.no_grad():
            shifts, cc, failed = AG.cc_search_shifts(s["vols"], s["targets"], s["ps"], case["width"],
                                                     case["max_shift"])
        return dict(shifts=shifts, cc=cc, failed=failed)
    vol, shifts = s["vol"].requires_grad_(True), s["shifts"].requires_grad_(True)
    vol.grad = shifts.grad = None
    images = AG.project(vol, shifts, s["setup"])
    (images - s["target"]).square().sum().backward()
    return dict(images=images, grad_volume=vol.grad, grad_shifts=shifts.grad)


# ------------------------------------------------------------------ work

def _chord(case, n_tilts):
    """Mean path of a ray through the volume's depth over the series, in voxels."""
    a = [math.radians(t) for t in (_tilt_angles(case) if n_tilts > 1 else [case["tilt"]])]
    return sum(1.0 / max(0.2, math.cos(t)) for t in a) / len(a)


def work(case):
    kind = case["kind"]
    # a ray's trilinear samples are summed cell by cell: about 30 operations a cell, 1.6 cells a layer;
    # a voxel's chord-weighted mean visits its OS^2 or more sub-rays at about 6 operations each
    if kind in ("operators", "sart", "sart_ctf", "project"):
        V, P = case["nx"] * case["ny"] * case["nz"], case["width"] * case["height"]
        T = case.get("tilts", 1)
        fp = 4 * P * 1.6 * case["nz"] * _chord(case, T) * 30.0
        if kind == "project":   # forward, its transpose and the shift derivative
            return dict(bytes=4.0 * (2 * V + 3 * T * P), flops=3.0 * T * fp)
        bp = V * (3.0 * case["os"] ** 2 * 6.0 + 10.0)
        vox = 2.0 if case.get("half") else 4.0
        S = case.get("sirt", 1)
        b = T * (vox * V * (1.0 + 2.0 / S) + 8.0 * P)
        f = T * (fp + bp)
        if kind == "sart_ctf":
            n = max(case["width"], case["height"])
            depth = np.mean([case["nz"] * math.cos(math.radians(t)) + case["nx"] * abs(math.sin(math.radians(t)))
                             for t in _tilt_angles(case)])
            slabs = depth * case["pixel_nm"] / case["slab_nm"]
            f += T * slabs * 4 * 2.5 * n * n * math.log2(n * n)
        return dict(bytes=b, flops=f)
    if kind == "subvol":
        c = case["cubes"]
        V = sum(c * r / 10.0 * n ** 3 for r, n in ((4, 32), (3, 64), (2, 96), (1, 128)))
        T, P = case["tilts"], case["width"] * case["height"]
        f = V * T * (3.0 * case["os"] ** 2 * 6.0 + 10.0)
        if case["ctf"]:
            n = max(case["width"], case["height"])
            depth = np.mean([case["depth"] * math.cos(math.radians(t)) + case["field"] * abs(math.sin(math.radians(t)))
                             for t in _tilt_angles(case)])
            f += T * (1 + depth / 16.0) * 2.5 * n * n * math.log2(n * n)
        return dict(bytes=8.0 * V + 4.0 * T * P, flops=f)
    if kind == "prep":
        P, n = case["width"] * case["height"], max(case["width"], case["height"])
        return dict(bytes=case["n"] * P * ((4 if case["dtype"] == "float32" else 2) + 4.0),
                    flops=case["n"] * (2 * 2.5 * n * n * math.log2(n * n) + 10.0 * n * n))
    n, K, T = case["n"], case["cubes"], case["tilts"]
    w = np.mean([n * (math.cos(math.radians(t)) + abs(math.sin(math.radians(t)))) for t in _tilt_angles(case)])
    pix = K * T * (w + 2 * case["margin"]) * (n + 2 * case["margin"])
    fp = 4 * K * T * n * w * 1.6 * n * 30.0
    if kind == "pair_grad":
        return dict(bytes=8.0 * K * n ** 3 + 12.0 * pix, flops=3.0 * fp)
    return dict(bytes=4.0 * K * n ** 3 + 12.0 * pix, flops=fp + pix * 2.0 * math.pi * case["max_shift"] ** 2)


# ------------------------------------------------------------------ exact values (float64, torch)

class _G:
    """Geometry as float64: the ray of pixel position (px, py) is d + xa u + ya v + t n."""

    def __init__(self, vg, tg):
        f = lambda a, n: [float(a[i]) for i in range(n)]  # noqa: E731
        self.d, self.u, self.v, self.n = f(tg.d, 3), f(tg.u, 3), f(tg.v, 3), f(tg.n, 3)
        self.M, self.A = f(tg.det_matrix, 16), f(tg.mag_aniso, 9)
        self.lo, self.hi = f(vg.bbox_min, 3), f(vg.bbox_max, 3)
        self.vs = f(vg.voxel_size, 3)
        self.scale = [float(vg.bbox_rcp[i]) * float(vg.dim[i]) for i in range(3)]
        self.zshift = float(vg.z_shift)
        self.size = (vg.nx, vg.ny, vg.nz)
        self.step = self.vs[0] * 0.15

    def origins(self, px, py, sx=0.0, sy=0.0):
        A_ = self.A
        xa = A_[0] * px + A_[1] * py + A_[2] - sx
        ya = A_[3] * px + A_[4] * py + A_[5] - sy
        return [self.d[i] + xa * self.u[i] + ya * self.v[i] for i in range(3)]

    def clip(self, c):
        """Entry and exit parameters of the rays, and the axis of the entry face."""
        t_in = torch.full_like(c[0], -math.inf)
        t_out = torch.full_like(c[0], math.inf)
        axis = torch.zeros_like(c[0], dtype=torch.long)
        for i in range(3):
            if self.n[i] == 0.0:
                inside = (c[i] >= self.lo[i]) & (c[i] <= self.hi[i])
                t_out = torch.where(inside, t_out, torch.full_like(t_out, -math.inf))
                continue
            a, b = (self.lo[i] - c[i]) / self.n[i], (self.hi[i] - c[i]) / self.n[i]
            lo = torch.minimum(a, b)
            axis = torch.where(lo > t_in, torch.full_like(axis, i), axis)
            t_in, t_out = torch.maximum(t_in, lo), torch.minimum(t_out, torch.maximum(a, b))
        return t_in, t_out, axis

    def texel(self, c, t):
        """Texel coordinates shifted so that texel j is centred at j."""
        return [(c[i] + t * self.n[i] - self.lo[i]) * self.scale[i] - 0.5 - (self.zshift if i == 2 else 0.0)
                for i in range(3)]


def _cell(g, q):
    """Clamp-addressed trilinear cell of texel coordinates: corner index, weights, unclamped axes."""
    i0, w, free = [], [], []
    for i in range(3):
        n = g.size[i]
        x = q[i].clamp(0.0, n - 1.0)
        k = x.floor().clamp(max=max(0, n - 2))
        i0.append(k.long())
        w.append(x - k)
        free.append(((q[i] >= 0.0) & (q[i] <= n - 1.0)).to(F64))
    nx, ny, _ = g.size
    return (i0[2] * ny + i0[1]) * nx + i0[0], w, free


def _corners(g):
    nx, ny, nz = g.size
    return [(dx, dy, dz, dz * nx * ny * (nz > 1) + dy * nx * (ny > 1) + dx * (nx > 1))
            for dz in (0, 1) for dy in (0, 1) for dx in (0, 1)]


def _trilinear(g, vol, q):
    o, w, _ = _cell(g, q)
    out = torch.zeros_like(w[0])
    for dx, dy, dz, off in _corners(g):
        out += vol[o + off] * (w[0] if dx else 1 - w[0]) * (w[1] if dy else 1 - w[1]) * (w[2] if dz else 1 - w[2])
    return out


def _sub_rays(W, H, x0, y0):
    y, x = torch.meshgrid(torch.arange(H, device=_device(), dtype=F64) + y0,
                          torch.arange(W, device=_device(), dtype=F64) + x0, indexing="ij")
    for ox in (0.25, 0.75):
        for oy in (0.25, 0.75):
            yield (x + ox).reshape(-1), (y + oy).reshape(-1)


_CHUNK = 1 << 22   # samples per torch operation


def _march(g, vol, W, H, x0=0, y0=0, shift=(0.0, 0.0), slab=None):
    """Projection and mean chord of the window; slab = (tmin, tmax) limits the samples to a CTF slab."""
    total = torch.zeros(W * H, device=_device(), dtype=F64)
    length, hits = torch.zeros_like(total), torch.zeros_like(total)
    for px, py in _sub_rays(W, H, x0, y0):
        c = g.origins(px, py, *shift)
        t_in, t_out, _ = g.clip(c)
        hit = t_out - t_in > 0.0
        length += torch.where(hit, t_out - t_in, torch.zeros_like(t_in))
        hits += hit.to(F64)
        first, last = t_in, t_out
        if slab is not None:
            first, last = t_in.clamp(min=slab[0]), t_out.clamp(max=slab[1])
            hit = hit & (first <= last)
            if not bool(hit.any()):
                continue
            # a slab's first sample is taken at the detector point
            total += torch.where(hit, _trilinear(g, vol, g.texel(c, torch.zeros_like(first))), torch.zeros_like(first))
            first = first + g.step
            hit = hit & (first <= last)
        idx = hit.nonzero().squeeze(1)
        if idx.numel() == 0:
            continue
        count = ((last[idx] - first[idx]) / g.step).floor() + 1.0
        q0 = g.texel([ci[idx] for ci in c], first[idx])
        dq = [g.step * g.n[i] * g.scale[i] for i in range(3)]
        most, per = int(count.max()), max(1, _CHUNK // idx.numel())
        acc = torch.zeros_like(count)
        for k0 in range(0, most, per):
            k = torch.arange(k0, min(most, k0 + per), device=_device(), dtype=F64)[None]
            val = _trilinear(g, vol, [q0[i][:, None] + k * dq[i] for i in range(3)])
            acc += (val * (k < count[:, None])).sum(1)
        total[idx] += acc
    return ((total * g.step * 0.25).reshape(H, W),
            torch.where(hits > 0, length / hits.clamp(min=1.0), torch.zeros_like(length)).reshape(H, W))


def _march_backward(g, vol, grad, W, H, gvol, x0=0, y0=0, shift=(0.0, 0.0)):
    """Adds the transpose of _march applied to grad (H, W) into gvol; returns the shift gradient."""
    gs = torch.zeros(2, device=_device(), dtype=F64)
    r = grad.reshape(-1) * (g.step * 0.25)
    for px, py in _sub_rays(W, H, x0, y0):
        c = g.origins(px, py, *shift)
        t_in, t_out, axis = g.clip(c)
        idx = (t_out - t_in > 0.0).nonzero().squeeze(1)
        if idx.numel() == 0:
            continue
        ri, first = r[idx], t_in[idx]
        count = ((t_out[idx] - first) / g.step).floor() + 1.0
        q0 = g.texel([ci[idx] for ci in c], first)
        dq = [g.step * g.n[i] * g.scale[i] for i in range(3)]
        most, per = int(count.max()), max(1, _CHUNK // idx.numel())
        G = [torch.zeros_like(first) for _ in range(3)]
        for k0 in range(0, most, per):
            k = torch.arange(k0, min(most, k0 + per), device=_device(), dtype=F64)[None]
            on = (k < count[:, None]).to(F64)
            o, w, free = _cell(g, [q0[i][:, None] + k * dq[i] for i in range(3)])
            for dx, dy, dz, off in _corners(g):
                f = [w[i] if (dx, dy, dz)[i] else 1 - w[i] for i in range(3)]
                gvol.index_add_(0, (o + off).reshape(-1), (f[0] * f[1] * f[2] * on * ri[:, None]).reshape(-1))
                v = vol[o + off] * on
                G[0] += (v * free[0] * (1 if dx else -1) * f[1] * f[2]).sum(1)
                G[1] += (v * free[1] * (1 if dy else -1) * f[0] * f[2]).sum(1)
                G[2] += (v * free[2] * (1 if dz else -1) * f[0] * f[1]).sum(1)
        ax = axis[idx]
        pick = lambda a: torch.as_tensor(a, device=_device(), dtype=F64)[ax]  # noqa: E731
        for j, e in enumerate((g.u, g.v)):   # a shift moves the samples by -e plus the entry point's slide
            slide = pick(e) / pick(g.n)
            gs[j] += sum((ri * G[i] * g.scale[i] * (-e[i] + slide * g.n[i])).sum() for i in range(3))
    return gs


def _centre_chord(g, W, H):
    y, x = torch.meshgrid(torch.arange(H, device=_device(), dtype=F64) + 0.5,
                          torch.arange(W, device=_device(), dtype=F64) + 0.5, indexing="ij")
    t_in, t_out, _ = g.clip(g.origins(x, y))
    return (t_out - t_in).clamp(min=0.0)


def _compare(real, virt, dist, length):
    return torch.where(dist >= 1.0, (real - virt / dist.clamp(min=1e-30) * length) / length, torch.zeros_like(virt))


def _crop_weight(W, H, p):
    """cropBorder's weight without dimming: 1 strictly inside the quadrilateral p1 p2 p4 p3."""
    y, x = torch.meshgrid(torch.arange(H, device=_device()), torch.arange(W, device=_device()), indexing="ij")
    (x1, y1), (x2, y2), (x3, y3), (x4, y4) = [(p[2 * i], p[2 * i + 1]) for i in range(4)]
    side = lambda ax, ay, bx, by: (bx - ax) * (y - ay) - (by - ay) * (x - ax) < 0  # noqa: E731
    return (side(x1, y1, x2, y2) & side(x4, y4, x3, y3) & side(x3, y3, x1, y1) & side(x2, y2, x4, y4)).to(F64)


def _bp(g, vol, img, lam, os, slabs=None):
    """vol (nz, ny, nx) += lam * chord-weighted mean of img over each voxel's sub-rays.  slabs = (starts,
    end of the last): img is a stack, and each voxel reads its slab's image with linear filtering."""
    nx, ny, nz = g.size
    H, W = img.shape[-2:]
    B = np.linalg.inv(np.array([g.u, g.v, g.n]).T)
    nn = math.sqrt(sum(x * x for x in g.n))
    n1 = [x / nn for x in g.n]
    M = g.M
    ext = [[0.0, 0.0], [0.0, 0.0]]   # projected box of a voxel relative to its corner
    for r in range(2):
        for i in range(3):
            e = B[r, i] * g.vs[i]
            ext[r][0] += min(0.0, e)
            ext[r][1] += max(0.0, e)
    points = [int(math.floor((ext[r][1] - ext[r][0]) * os)) + 2 for r in range(2)]
    nd = -sum(g.n[i] * g.d[i] for i in range(3))
    for z0 in range(0, nz, max(1, _CHUNK // (nx * ny))):
        z1 = min(nz, z0 + max(1, _CHUNK // (nx * ny)))
        z, y, x = torch.meshgrid(torch.arange(z0, z1, device=_device(), dtype=F64),
                                 torch.arange(ny, device=_device(), dtype=F64),
                                 torch.arange(nx, device=_device(), dtype=F64), indexing="ij")
        xq = (x / 4).floor() * 4
        base = [g.lo[0] + xq * g.vs[0], g.lo[1] + y * g.vs[1], g.lo[2] + z * g.vs[2]]
        far = [g.lo[0] + (xq + 5) * g.vs[0], g.lo[1] + (y + 1) * g.vs[1], g.lo[2] + (z + 1) * g.vs[2]]
        lo = hi = ok = None
        for corner in range(8):
            c = [far[i] if corner >> (2 - i) & 1 else base[i] for i in range(3)]
            t = (g.n[0] * c[0] + g.n[1] * c[1] + g.n[2] * c[2] + nd).abs()
            if corner == 0 and slabs is None:
                ok = t < 9999999999999.0
            elif corner == 0:
                starts = torch.as_tensor([float(v) for v in slabs[0]], device=_device(), dtype=F64)
                slab = (torch.searchsorted(starts, t.contiguous(), right=True) - 1)
                ok = (slab >= 0) & (t < float(slabs[1]))
                slab = slab.clamp(min=0)
            h = [c[i] - t * g.n[i] for i in range(3)]
            lo = h if lo is None else [torch.minimum(a, b) for a, b in zip(lo, h)]
            hi = h if hi is None else [torch.maximum(a, b) for a, b in zip(hi, h)]
        if not bool(ok.any()):
            continue
        if g.n[0] <= 0.0:
            lo[0], hi[0] = hi[0], lo[0]
        b0, b1 = [], []
        for r in range(2):
            f = lambda p: M[4 * r] * p[0] + M[4 * r + 1] * p[1] + M[4 * r + 2] * p[2] + M[4 * r + 3]  # noqa: E731
            a, b = f(lo), f(hi)
            lim = (W if r == 0 else H) - 1
            b0.append(torch.minimum(a, b).floor().clamp(0, lim) * os)
            b1.append(torch.maximum(a, b).ceil().clamp(0, lim) * os)
        corner = [g.lo[0] + x * g.vs[0] - g.d[0], g.lo[1] + y * g.vs[1] - g.d[1], g.lo[2] + z * g.vs[2] - g.d[2]]
        P = [sum(B[r, i] * corner[i] for i in range(3)) for r in range(2)]
        start = [((P[r] + ext[r][0]) * os - 0.5).floor() for r in range(2)]
        num, den = torch.zeros_like(x), torch.zeros_like(x)
        for dj in range(points[1]):
            jj = start[1] + dj
            for di in range(points[0]):
                ii = start[0] + di
                on = ok & (ii >= b0[0]) & (ii < b1[0]) & (jj >= b0[1]) & (jj < b1[1])
                pu, pv = (ii + 0.5) / os, (jj + 0.5) / os
                a, b = pu - P[0], pv - P[1]
                t_in = torch.full_like(a, -math.inf)
                t_out = torch.full_like(a, math.inf)
                for i in range(3):
                    w = a * g.u[i] + b * g.v[i]
                    if abs(n1[i]) < 1e-6:
                        on = on & (w > 0.0) & (w < g.vs[i])
                        continue
                    e, f = -w / n1[i], (g.vs[i] - w) / n1[i]
                    t_in, t_out = torch.maximum(t_in, torch.minimum(e, f)), torch.minimum(t_out, torch.maximum(e, f))
                chord = torch.where(on, (t_out - t_in).clamp(min=0.0), torch.zeros_like(a))
                if slabs is not None:
                    xb, yb = pu - 0.5, pv - 0.5
                    x0, y0 = xb.floor(), yb.floor()
                    wx, wy = xb - x0, yb - y0
                    at = lambda i, j: img[slab, j.clamp(0, H - 1).long(), i.clamp(0, W - 1).long()]  # noqa: E731
                    val = ((at(x0, y0) * (1 - wx) + at(x0 + 1, y0) * wx) * (1 - wy)
                           + (at(x0, y0 + 1) * (1 - wx) + at(x0 + 1, y0 + 1) * wx) * wy)
                else:
                    val = img[pv.floor().clamp(0, H - 1).long(), pu.floor().clamp(0, W - 1).long()]
                num += val * chord
                den += chord
        vol[z0:z1] += torch.where(den > 0, lam * num / den.clamp(min=1e-300), torch.zeros_like(num))


def _f32(x):
    return float(np.float32(x))


def _slabs(rng_, ctf):
    """Slab starts as the float loop steps them, and the step."""
    step = np.float32(ctf.slice_thickness_nm) / np.float32(ctf.pixelsize_nm)
    out, ray = [], np.float32(rng_[0])
    while ray < np.float32(rng_[1]):
        out.append(ray)
        ray = np.float32(ray + step)
    return out, step


def _slab_defocus(ray, d, ctf):
    """Defocus range of a slab (nm), in single precision: the values that enter the CTF."""
    f = np.float32
    T = f(ctf.slice_thickness_nm)
    prod = f(f(f(ray) + f(-10000.0)) * f(ctf.pixelsize_nm)) * T
    z = f(f(math.copysign(math.floor(abs(float(prod)) + 0.5), float(prod))) / T) + T / f(2.0)
    tilt = f(f(f(d.tilt_deg) / f(180.0)) * f(math.pi))
    z = z - f(f(f(ctf.volume_shift_z) * f(ctf.pixelsize_nm)) * f(np.cos(tilt)))
    return f(f(d.defocus_min_nm) + z), f(f(d.defocus_max_nm) + z)


def _ctf_filter(square, ctf, dmin, dmax, angle_deg, forward):
    N = square.shape[0]
    f = np.float32
    pi = f(math.pi)
    kV = f(ctf.voltage_kV)
    a = f(f(f(f(2 * 511) * kV) * f(1000)) * f(1000)) + f(f(f(kV * kV) * f(1000)) * f(1000))
    lam = float(f(f(6.63e-34) * f(3.0e8)) / np.sqrt(f(float(a) * 1.602e-19 * 1.602e-19)))
    ps = f(ctf.pixelsize_nm) * f(10.0) ** f(-9.0)
    freq = float(f(1.0 / float(f(ps * f(2.0)))) / (f(N) / f(2.0)))
    cs, ac = float(f(ctf.cs_mm) * f(0.001)), float(ctf.amp_contrast)
    pc = float(np.sqrt(f(1) - f(ac) * f(ac)))
    d0, d1 = float(f(dmin) * f(0.000000001)), float(f(dmax) * f(0.000000001))
    y = torch.arange(N, device=_device(), dtype=F64)[:, None]
    y = torch.where(y > N * 0.5, y - N, y)
    x = torch.arange(N // 2 + 1, device=_device(), dtype=F64)[None].expand(N, -1)
    alpha = torch.where(x == 0, torch.full_like(x, float(pi * f(0.5))), torch.atan2(y.expand_as(x), x))
    defocus = d0 + (1 - torch.cos(2 * (alpha - float(f(f(angle_deg) / f(180.0)) * pi)))) * (d1 - d0)
    radius = torch.sqrt(x * x + y * y)
    k = radius * freq
    m = float(pi / f(2.0)) * (cs * lam ** 3 * k ** 4 - 2 * defocus * lam * k * k)
    n = pc * torch.sin(m) + ac * torch.cos(m)
    beta = [float(ctf.beta_fac[i]) for i in range(4)]
    e = k / 1e8
    env = torch.exp((-beta[1] * e - beta[2] * e * e) - beta[3] * e ** 3)
    if forward:
        val = n * env.clamp(min=_f32(0.01))
        tiny = _f32(0.0001)
        val = torch.where(val.abs() < tiny, torch.where(val >= 0, torch.full_like(val, tiny),
                                                        torch.full_like(val, -tiny)), val)
        fac = -val
    else:
        val = n * env.clamp(min=float(ctf.wiener))
        fac = -val / (val * val + float(ctf.wiener))
    fac = torch.where(radius > beta[0], fac, torch.ones_like(fac))
    return torch.fft.irfft2(torch.fft.rfft2(square) * fac, s=(N, N))


def _filtered(img, weight, ctf, dmin, dmax, angle, forward):
    H, W = img.shape
    N = max(W, H)
    bx, by = (N - W) // 2, (N - H) // 2
    sq = torch.zeros((N, N), device=_device(), dtype=F64)
    sq[by:by + H, bx:bx + W] = img
    out = _ctf_filter(sq, ctf, dmin, dmax, angle, forward)[by:by + H, bx:bx + W]
    return out if weight is None else out * weight


def _exact_sart(case, seed):
    s = _sart_inputs(case, seed)
    vg, acq, sp = s["vg"], s["acq"], s["sp"]
    W, H, S = case["width"], case["height"], case["sirt"]
    vol = torch.zeros((vg.nz, vg.ny, vg.nx), device=_device(), dtype=F64)
    lam = _f32(np.float32(sp.lambda_) / np.float32(S))
    T, empty = len(acq.geoms), True
    frame = _crop_weight(W, H, [0, H - 1, W - 1, H - 1, 0, 0, W - 1, 0])
    for s0 in range(0, T, S):
        subset = acq.index_list[s0:s0 + S]
        resid = []
        for i in subset:
            g = _G(vg, acq.geoms[i])
            virt, dist = torch.zeros((H, W), device=_device(), dtype=F64), None
            if not empty and case["kind"] == "sart":
                virt, dist = _march(g, vol.reshape(-1), W, H)
            elif not empty:
                starts, step = _slabs(acq.slab_ranges[i], s["ctf"])
                for ray in starts:
                    img, _ = _march(g, vol.reshape(-1), W, H, slab=(float(ray), float(np.float32(ray + step))))
                    dmin, dmax = _slab_defocus(ray, s["defocus"][i], s["ctf"])
                    virt = virt + _filtered(img * frame, frame, s["ctf"], dmin, dmax,
                                            s["defocus"][i].astig_angle_deg, True)
            if dist is None:
                dist = _centre_chord(g, W, H)
            resid.append(_compare(s["projs"][i].to(F64), virt, dist, float(acq.real_lengths[i])))
        for i, r in zip(subset, resid):
            g, w = _G(vg, acq.geoms[i]), _crop_weight(W, H, acq.hitpoints[i])
            if case["kind"] == "sart":
                _bp(g, vol, r * w, lam, case["os"])
                continue
            starts, step = _slabs(acq.slab_ranges[i], s["ctf"])
            stack = []
            for ray in starts:
                dmin, dmax = _slab_defocus(ray, s["defocus"][i], s["ctf"])
                stack.append(_filtered(r * w, w, s["ctf"], dmin, dmax, s["defocus"][i].astig_angle_deg, False))
            _bp(g, vol, torch.stack(stack), lam, case["os"], (starts, starts[-1] + step))
        empty = False
        if case.get("half"):
            vol = vol.to(torch.float16).to(F64)
    return dict(volume=vol)


def _exact_operators(case, seed):
    vg, acq, projs, d = _series(case, seed)
    W, H = case["width"], case["height"]
    g = _G(vg, acq.geoms[0])
    proj, dist = _march(g, _density_volume(d, vg).to(F64).reshape(-1), W, H)
    r = _compare(projs[0].to(F64), proj, dist, float(acq.real_lengths[0])) * _crop_weight(W, H, acq.hitpoints[0])
    upd = torch.zeros((vg.nz, vg.ny, vg.nx), device=_device(), dtype=F64)
    _bp(g, upd, r, _f32(0.3), case["os"])
    return dict(residual=r, dist=dist, update=upd)


def _exact_subvol(case, seed):
    s = _subvol_inputs(case, seed)
    out = [torch.zeros((v.nz, v.ny, v.nx), device=_device(), dtype=F64) for v in s["vgs"]]
    for t in range(case["tilts"]):
        img = s["images"][t].to(F64)
        if not case["ctf"]:
            for v, g, o in zip(s["vgs"], s["geoms"], out):
                _bp(_G(v, g[t]), o, img, 1.0, case["os"])
            continue
        kw = s["kw"]
        starts, step = _slabs(kw["slab_ranges"][t], kw["ctf"])
        stack = torch.empty((len(starts),) + tuple(img.shape), device=_device(), dtype=F64)
        for k, ray in enumerate(starts):
            dmin, dmax = _slab_defocus(ray, kw["defocus"][t], kw["ctf"])
            stack[k] = _filtered(img, None, kw["ctf"], dmin, dmax, kw["defocus"][t].astig_angle_deg, False)
        for v, g, o in zip(s["vgs"], s["geoms"], out):
            _bp(_G(v, g[t]), o, stack, 1.0, case["os"], (starts, starts[-1] + step))
    return dict(cubes=torch.cat([o.reshape(-1) for o in out]))


def _mirror(img, N):
    H, W = img.shape
    def src(n, b):  # noqa: E306
        i = torch.arange(N, device=img.device) - b
        i = torch.where(i < 0, -i - 1, i)
        i = torch.where(i >= n, 2 * n - i - 1, i)
        return i.clamp(0, n - 1)
    return img[src(H, (N - H) // 2)][:, src(W, (N - W) // 2)]


def _exact_prep(case, seed):
    s = _prep_inputs(case, seed)
    W, H = case["width"], case["height"]
    N = max(W, H)
    bx, by = (N - W) // 2, (N - H) // 2
    y = torch.arange(N, device=_device(), dtype=F64)[:, None]
    y = torch.where(y > N * 0.5, y - N, y)
    x = torch.arange(N // 2 + 1, device=_device(), dtype=F64)[None]
    dist = torch.sqrt(x * x + y * y)
    lp, lps = _f32(s["common"]["lp"]), _f32(s["common"]["lps"])
    lp = _f32(np.float32(lp) - np.float32(lps))
    fil = (dist <= lp).to(F64)
    soft = (1.0 - fil) * torch.exp(-((dist - lp) ** 2 / (2 * lps * lps)))
    fil = torch.where(soft > _f32(0.001), soft, fil)
    out = torch.empty((case["n"], H, W), device=_device(), dtype=F64)
    mean, std = [], []
    for i in range(case["n"]):
        img = s["images"][i]
        img = (img.view(torch.int16) if img.dtype == torch.uint16 else img).to(F64)   # counts stay below 2^15
        sq = _mirror(img, N)
        m = float(np.float32(float(sq.mean())))
        sq = torch.where(sq > _f32(np.float32(10.0) * np.float32(m)), torch.full_like(sq, m), sq)
        if case["wbp"]:
            raw = sq[by:by + H, bx:bx + W]
            mean.append(_f32(float(raw.mean())))
            std.append(_f32(float(raw.std(unbiased=False))))
            raw = ((raw - mean[-1]) / -std[-1])
            sq = _mirror(raw, N)
        X = torch.fft.rfft2(sq) * fil
        if case["wbp"]:
            ang = float(np.float32(-np.float32(s["psis"][i])) / np.float32(180.0) * np.float32(math.pi))
            X = X * ((math.sin(ang) * x + math.cos(ang) * y) / N / 2.0).abs().clamp(max=1.0)
        else:
            X = X * torch.exp(-_f32(s["dose"][i]) * (dist / (N // 2 / _f32(2.5))))
        res = torch.fft.irfft2(X, s=(N, N))[by:by + H, bx:bx + W]
        if not case["wbp"]:
            mean.append(_f32(float(res.mean())))
            std.append(_f32(float(res.std(unbiased=False))))
            res = (res - mean[-1]) / -mean[-1]
        out[i] = res
    return dict(out=out, mean=np.array(mean), std=np.array(std), bad=None)


def _exact_pairs(case, seed):
    s = _pair_inputs(case, seed)
    vols, n3 = s["vols"].to(F64), case["n"] ** 3
    targets = s["targets"].to(F64)
    images, gvol, gshift, peaks, ccs, off = [], torch.zeros_like(vols), [], [], [], 0
    for (k, x0, y0, w, h), tg in zip(s["pairs"], s["geoms"]):
        g, vol = _G(s["subs"][k][0], tg), vols[k * n3:(k + 1) * n3]
        img, _ = _march(g, vol, w, h, x0, y0)
        target = targets[off:off + w * h].reshape(h, w)
        off += w * h
        if case["kind"] == "pair_grad":
            images.append(img.reshape(-1))
            gshift.append(_march_backward(g, vol, 2.0 * (img - target), w, h, gvol[k * n3:(k + 1) * n3], x0, y0))
            continue
        N, m = float(case["width"]), case["max_shift"]
        side = 2 * m + 1
        pad = torch.nn.functional.pad(target, (m, m, m, m))
        corr = torch.empty((side, side), device=_device(), dtype=F64)
        for ry in range(-m, m + 1):
            for rx in range(-m, m + 1):
                corr[ry + m, rx + m] = (img * pad[m - ry:m - ry + h, m - rx:m - rx + w]).sum()
        sa, sb = target.sum(), img.sum()
        den = torch.sqrt((target.square().sum() - sa * sa / N ** 2) * (img.square().sum() - sb * sb / N ** 2))
        r = torch.arange(-m, m + 1, device=_device(), dtype=F64)
        cc = torch.where(r[:, None] ** 2 + r[None] ** 2 <= m * m, (corr - sa * sb / N ** 2) / den,
                         torch.full_like(corr, -math.inf))
        best = int(cc.argmax())
        ccs.append(float(cc.reshape(-1)[best]))
        peaks.append((-(best % side - m), -(best // side - m)))
    if case["kind"] == "pair_grad":
        return dict(images=torch.cat(images), grad_volumes=gvol, grad_shifts=torch.stack(gshift))
    return dict(shifts=torch.tensor(peaks, dtype=F64), cc=torch.tensor(ccs, dtype=F64), failed=None)


def _exact_project(case, seed):
    s = _project_inputs(case, seed)
    vg, W, H = s["vg"], case["width"], case["height"]
    vol = s["vol"].to(F64).reshape(-1)
    acq, gvol, images, gs = s["acq"], torch.zeros_like(vol), [], []
    for t, (tilt, psi) in enumerate(zip(acq.tilts_deg, acq.psis_deg)):
        e = s["shifts"][t].tolist()
        g = _G(vg, A.subvolume_tilt_geometry(tilt, W, H, psi_deg=psi, extra_shift=e))
        img, _ = _march(g, vol, W, H)
        images.append(img)
        gs.append(_march_backward(g, vol, 2.0 * (img - s["target"][t].to(F64)), W, H, gvol))
    return dict(images=torch.stack(images), grad_volume=gvol.reshape(vg.nz, vg.ny, vg.nx), grad_shifts=torch.stack(gs))


def _samples(case):
    """About how many ray samples (forward and backward ones counted alike) `exact` evaluates."""
    if case["kind"] in ("pair_grad", "pair_search"):
        return work(dict(case, kind="pair_search", max_shift=0))["flops"] / 30.0 * 4.2 * (
            6.0 if case["kind"] == "pair_grad" else 1.0)
    T = case.get("tilts", 1)
    return 4.0 * case["width"] * case["height"] * case["nz"] * _chord(case, T) * T * 6.7 * (
        6.0 if case["kind"] == "project" else 1.0)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "operators":
            return _exact_operators(case, seed)
        if kind == "prep":
            return _exact_prep(case, seed)
        if kind == "subvol":
            c, T = case["cubes"], case["tilts"]
            V = c * (0.4 * 32 ** 3 + 0.3 * 64 ** 3 + 0.2 * 96 ** 3 + 0.1 * 128 ** 3)
            return None if V * T > 1.5e9 or c * T > 1200 else _exact_subvol(case, seed)
        if kind == "pair_search" and case["cubes"] * case["tilts"] * (2 * case["max_shift"] + 1) ** 2 > 4e5:
            return None   # one torch call per candidate shift
        pairs = case["cubes"] * case["tilts"] if kind.startswith("pair") else 0
        if _samples(case) > 2.5e10 or pairs > 600:
            return None
        if kind in ("sart", "sart_ctf"):
            return _exact_sart(case, seed)
        if kind == "project":
            return _exact_project(case, seed)
        return _exact_pairs(case, seed)


__all__ = ["draw", "exact", "listed", "prepare", "run", "work"]
