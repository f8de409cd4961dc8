"""GPU checks of the walk of rays without a y component (tilts about y) at the sizes where it can go
wrong: volumes of one layer more or less than a slab, two voxels on an axis, widths that leave tile
remainders, both ray directions, and sub-volumes at the limits of the LDS planes of the pair adjoint.

The transposes are checked with all-positive inputs, so that the two sums of <P x, y> = <x, P^T y> do not
cancel: each is a sum of float-rounded positive terms (relative error 2^-24 per projection pixel and per
gradient voxel, and the per-cell rounding 2^-24 of the projector), so they agree within 4 * 2^-24 = 2.4e-7;
the bound is twice that."""
import numpy as np
import pytest
import torch

import artiatomi_amd as A

pytestmark = pytest.mark.gpu

BOUND = 5e-7


@pytest.fixture(scope="module")
def ctx(gpu):
    c = A.ArtiaContext(0)
    yield c
    c.set_fp_staging(True)
    c.close()


def positive(shape, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return 0.5 + torch.rand(shape, generator=gen, device="cuda")


SIZES = [
    # (nx, ny, nz, W, H, tilt, psi)
    (4, 2, 2, 9, 7, 10.0, 0.0),
    (8, 9, 7, 17, 15, -31.0, 0.0),
    (12, 8, 8, 8, 8, 60.0, 5.0),
    (20, 17, 9, 31, 33, -60.0, -5.0),
    (64, 33, 15, 70, 41, 0.0, 0.0),
    (64, 40, 17, 65, 57, 44.0, 90.0),
    (36, 36, 33, 50, 50, -12.0, 41.0),
]


@pytest.mark.parametrize("nx,ny,nz,W,H,tilt,psi", SIZES)
def test_flat_walk_staged_equals_direct_and_transpose(ctx, nx, ny, nz, W, H, tilt, psi):
    print(f"flat walk {nx}x{ny}x{nz} -> {W}x{H}, tilt {tilt} psi {psi}", flush=True)
    vg = A.volume_geometry(nx, ny, nz)
    g = A.tilt_geometry(tilt, W, H, psi_deg=psi, shift=(0.4, -0.7))
    x, y = positive((nz, ny, nx), 1), positive((H, W), 2)
    proj, grad = [], []
    for staged in (True, False):
        ctx.set_fp_staging(staged)
        p, d = torch.zeros((H, W), device="cuda"), torch.zeros((H, W), device="cuda")
        ctx.fp_march(vg, g, x, p, d)
        gv = torch.zeros_like(x)
        ctx.fp_adjoint(vg, g, y, gv)
        proj.append(p)
        grad.append(gv)
    assert float(proj[0].max()) > 0
    assert torch.equal(proj[0], proj[1])
    lhs = float((proj[0].double() * y.double()).sum())
    for gv in grad:
        rhs = float((x.double() * gv.double()).sum())
        assert abs(lhs - rhs) <= BOUND * abs(lhs), abs(lhs - rhs) / abs(lhs)


@pytest.mark.parametrize("n", [16, 40, 64, 96, 104])
@pytest.mark.parametrize("psi", [0.0, 4.0, 33.0, 87.0])
def test_pair_adjoint_is_the_transpose(ctx, n, psi):
    """Eight planes of rows in LDS (16), as many as fit (40, 64, 96: two) and the form beyond (104);
    lanes along either detector axis."""
    print(f"pair adjoint {n}^3 psi {psi}", flush=True)
    full = A.volume_geometry(256, 256, 128)
    vols, subs, pairs, geoms = positive((2, n, n, n), 3), [], [], []
    for k, pos in enumerate(((100.3, 120.0, 60.0), (140.0, 131.7, 66.2))):
        vg = A.subvolume_geometry(n, 1.0, (1.0, 1.0, 1.0), full, pos)
        subs.append((vg, k * n ** 3))
        for tilt in (-57.0, 0.0, 21.0):
            g = A.tilt_geometry(tilt, 256, 256, psi_deg=psi)
            x0, y0, w, h = A.footprint_window(vg, g, 256, 256, 3)
            pairs.append((k, x0, y0, w, h))
            geoms.append(g)
    ps = A.PairSet(ctx, subs, pairs, geoms)
    flat = vols.reshape(-1).contiguous()
    shifts = torch.as_tensor(np.random.default_rng(4).uniform(-2, 2, (ps.npairs, 2)), device="cuda")
    images = positive(ps.n_pixels, 5)
    grad = torch.zeros_like(flat)
    ps.adjoint(shifts, images, grad)
    lhs = float((ps.project(flat, shifts).double() * images.double()).sum())
    rhs = float((grad.double() * flat.double()).sum())
    assert abs(lhs - rhs) <= BOUND * abs(lhs), abs(lhs - rhs) / abs(lhs)
    ps.close()


@pytest.mark.parametrize("n", [16, 40, 64, 94, 95])
@pytest.mark.parametrize("psi", [0.0, 2.0, 4.0, 10.0, 33.0, -45.0, 87.0, -88.0, 135.0])
def test_staged_pair_adjoint_is_the_transpose(ctx, n, psi):
    """The same from runs of y rows in LDS: eight planes of rows (16, 40), four (64), the last size with two (94)
    and the first without (95); runs along a detector axis, wider and narrower than a window, and oblique."""
    ctx.set_fp_staging(True)
    test_pair_adjoint_is_the_transpose(ctx, n, psi)


def march_given_samples(vg, g, vol, W, H):
    """Projection in float64 at the walk's own sample lattice: its float start and step of every sub-ray."""
    f = lambda a: np.array(list(a), np.float64)  # noqa: E731
    n, u, v, d, lo, hi = f(g.n), f(g.u), f(g.v), f(g.d), f(vg.bbox_min), f(vg.bbox_max)
    scale, size, a = f(vg.bbox_rcp) * f(vg.dim), (vg.nx, vg.ny, vg.nz), f(g.mag_aniso)
    step = float(vg.voxel_size[0]) * 0.15
    dq = (step * n * scale).astype(np.float32).astype(np.float64)
    total = torch.zeros((H, W), dtype=torch.float64, device="cuda")
    py, px = np.mgrid[0:H, 0:W]
    for ox in (0.25, 0.75):
        for oy in (0.25, 0.75):
            x, y = px + ox, py + oy
            xa, ya = a[0] * x + a[1] * y + a[2], a[3] * x + a[4] * y + a[5]
            c = d + xa[..., None] * u + ya[..., None] * v
            with np.errstate(divide="ignore", invalid="ignore"):
                t = np.stack([(lo - c) / n, (hi - c) / n])
            t_in, t_out = np.nanmin(t, 0).max(-1), np.nanmax(t, 0).min(-1)
            count = np.where(t_out > t_in, np.floor((t_out - t_in) / step) + 1.0, 0.0)
            q0 = (c + np.where(count > 0, t_in, 0.0)[..., None] * n - lo) * scale - 0.5
            q0[..., 2] -= float(vg.z_shift)
            q0 = torch.from_numpy(q0.astype(np.float32).astype(np.float64)).cuda()
            k = torch.arange(int(count.max()), dtype=torch.float64, device="cuda")
            val, off = torch.ones((H, W, len(k)), dtype=torch.float64, device="cuda"), []
            for i in range(3):
                q = q0[..., i, None] + k * dq[i]
                j = q.floor()
                off.append((j.long().clamp(0, size[i] - 1), (j.long() + 1).clamp(0, size[i] - 1), q - j))
            val = 0.0
            for cz in (0, 1):
                for cy in (0, 1):
                    for cx in (0, 1):
                        w = 1.0
                        for (o, s) in zip(off, (cx, cy, cz)):
                            w = w * (o[2] if s else 1.0 - o[2])
                        val = val + w * vol[off[2][cz], off[1][cy], off[0][cx]].double()
            total += (val * (k < torch.from_numpy(count).cuda()[..., None])).sum(-1)
    return total * (step * 0.25)


@pytest.mark.parametrize("staged", [True, False])
def test_flat_walk_keeps_its_position(ctx, staged):
    """Waves of 8 voxels whose fronts hold the rays: a shift of the samples by e voxels across the rays, which all
    rays of one entry face share, changes the projection by up to 0.8 e.  The walk's middles carry two roundings of
    values below 1 and of lo, 1.3e-7 in all, and the pixel its own 6e-8: gate 2e-7.  (A position kept in one float
    lost up to 4e-6 over the 90 layers of each ray.)"""
    nx, ny, nz, W, H = 128, 6, 96, 130, 6
    vg, g = A.volume_geometry(nx, ny, nz), A.tilt_geometry(43.0, W, H)
    n = np.array(list(g.n), np.float64)
    z, x = np.mgrid[0:nz, 0:nx].astype(np.float64)
    front = 1.0 + 0.9 * np.sin(2.0 * np.pi / 8.0 * (x * n[2] - z * n[0]) / np.hypot(n[0], n[2]))
    vol = torch.from_numpy(np.repeat(front[:, None], ny, 1).astype(np.float32)).cuda().contiguous()
    ref = march_given_samples(vg, g, vol, W, H)
    ctx.set_fp_staging(staged)
    p, d = torch.zeros((H, W), device="cuda"), torch.zeros((H, W), device="cuda")
    ctx.fp_march(vg, g, vol, p, d)
    err = float((p.double() - ref).norm() / ref.norm())
    print(f"flat position staged {staged}: {err:.2e}", flush=True)
    assert err <= 2e-7


def test_direct_walk_reads_infinite_voxels_only_at_samples(ctx):
    """From memory, a ray that crosses a cell between two of its samples takes nothing from it: exactly the pixels
    with a sample beside an infinite voxel are not finite."""
    nx, ny, nz, W, H = 64, 40, 40, 90, 42
    vg, vol = A.volume_geometry(nx, ny, nz), positive((nz, ny, nx), 12)
    at = np.random.default_rng(6).integers([4, 2, 4], [36, 38, 60], (60, 3))
    vol[at[:, 0], at[:, 1], at[:, 2]] = float("inf")
    ctx.set_fp_staging(False)
    for tilt in (61.0, -34.0, 17.0):
        g = A.tilt_geometry(tilt, W, H, shift=(0.3, 0.2))
        p, d = torch.zeros((H, W), device="cuda"), torch.zeros((H, W), device="cuda")
        ctx.fp_march(vg, g, vol, p, d)
        ref = march_given_samples(vg, g, vol, W, H)
        assert 0 < int((~ref.isfinite()).sum()) < W * H // 2
        assert torch.equal(p.isfinite(), ref.isfinite()), tilt
