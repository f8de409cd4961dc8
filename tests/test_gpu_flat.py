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
