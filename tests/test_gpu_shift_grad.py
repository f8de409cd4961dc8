"""fp_shift_grad through LDS-staged slabs against its direct walk, at the sizes where tiles, slabs and boxes
leave remainders, for rays without a y component and (a declined beam) with one.

Both add the same per-sub-ray doubles; only the order of the blocks' sums differs.  The volume rises along
every axis and the gradient image is positive, so a component's terms have one sign but for the volume's
faces: gate 1e-10 of the larger component (some 1e4 sums of relative error 2^-53 each)."""
import pytest
import torch

import artiatomi_amd as A
from artiatomi_amd._abi import GlobalParams
from test_gpu_flat import SIZES, positive

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam", [0.0, 7.0])
@pytest.mark.parametrize("nx,ny,nz,W,H,tilt,psi", SIZES)
def test_staged_equals_direct(gpu, nx, ny, nz, W, H, tilt, psi, beam):
    print(f"shift gradient {nx}x{ny}x{nz} -> {W}x{H}, tilt {tilt} psi {psi} beam {beam}", flush=True)
    vg = A.volume_geometry(nx, ny, nz)
    glob = GlobalParams(0.0, 0.0, beam, 0, 0.0)
    g = A.tilt_geometry(tilt, W, H, psi_deg=psi, shift=(0.4, -0.7), glob=glob)
    assert (abs(g.n[1]) > 1e-3) == (beam != 0.0 and tilt != 0.0)
    z, y, x = torch.meshgrid(*(torch.arange(n, device="cuda", dtype=torch.float32) for n in (nz, ny, nx)), indexing="ij")
    vol = (x + 2.0 * y + 4.0 * z + positive((nz, ny, nx), 5)).contiguous()
    gout = positive((H, W), 6)
    res = []
    ctx = A.ArtiaContext(0)
    try:
        for staged in (True, False):
            ctx.set_fp_staging(staged)
            for roi in (None, (1, 2, W - 1, H - 2)):
                out = torch.zeros(2, dtype=torch.float64, device="cuda")
                ctx.fp_shift_grad(vg, g, vol, gout, out, roi=roi)
                res.append(out.cpu())
    finally:
        ctx.close()
    for a, b in zip(res[:2], res[2:]):
        assert float(a.abs().max()) > 0
        assert float((a - b).abs().max()) <= 1e-10 * float(a.abs().max())
