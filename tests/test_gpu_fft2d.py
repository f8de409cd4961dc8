"""The three-kernel Fourier filters at each supported square (N = 128 .. 4096, a power of two) and at
images that fill it, leave ragged borders or are much narrower, against the FP64 compositions.

Tolerance: a transform's rounding errors are independent over its log2 N^2 <= 24 radix-2 levels, about
0.6 u each (u = 2^-24) with as much again from the rounded twiddles, so one direction carries
0.6 u sqrt(2 * 24) = 2.5e-7 and forward and back 3.5e-7 relative L2 for white images; gate 1e-6.
"""
import numpy as np
import pytest
import torch

import artiatomi_amd as A
import ctf_compose as CC
import oracle_lib as O
import prep_compose as P
from conftest import rel_l2
from test_gpu_ctf import per_slab_sart_ctf

pytestmark = pytest.mark.gpu

SIZES = [(128, 128), (127, 128), (128, 5), (256, 201), (512, 512), (333, 512), (1024, 1022), (2048, 1111), (4096, 64),
         (2047, 4096)]


@pytest.fixture(scope="module")
def ctx(gpu):
    c = A.ArtiaContext(0)
    yield c
    c.close()


def white(H, W, seed):
    return np.random.default_rng(seed).standard_normal((H, W)).astype(np.float32)


def mirror_square(img, N):
    """Mirror padding, clamped where a pad is wider than the image (the oracle's is not defined there)."""
    def index(n):
        i = np.arange(N) - (N - n) // 2
        i = np.where(i < 0, -i - 1, i)
        return np.clip(np.where(i >= n, 2 * n - i - 1, i), 0, n - 1)

    return img[np.ix_(index(img.shape[0]), index(img.shape[1]))]


@pytest.mark.parametrize("W,H", SIZES)
def test_slab_and_wbp_filters(ctx, W, H):
    print(f"filters {W} x {H}", flush=True)
    img, base = white(H, W, W + H), white(H, W, 1)
    N = max(W, H)
    corners = [0, H - 1, W - 1, H - 1, 0, 0, W - 1, 0]
    p = A.ctf_params(pixelsize_nm=0.5, beta_fac=(2.0, 0.0, 0.008, 0.0), amp_contrast=0.07)
    k = O.ctf_consts(2.7, 300.0, 0.5, N, 0.07)
    for for_fp, cut, dim in ((True, (0.0, 0.0), (2.0, 2.0)), (False, (1.0, 0.0), (1.0, 1.0))):
        d_img, d_out = torch.from_numpy(img).cuda(), torch.from_numpy(base).cuda()
        ctx.ctf_slab_filter(d_img, d_out, corners, p, 3000.0, 3150.0, 20.0, for_fp=for_fp, accumulate=for_fp,
                            cut_length=cut, dim_length=dim)
        _, f = CC.slab_filter(img.astype(np.float64), corners, k, 3000.0, 3150.0, 20.0, for_fp, cut, dim,
                              beta=tuple(p.beta_fac))
        expect = base.astype(np.float64) + f if for_fp else f
        assert float(np.abs(f).max()) > 0
        assert rel_l2(d_out.cpu().numpy(), expect) <= 1e-6
    out = torch.zeros((H, W), device="cuda")
    for method in ("ramp", "contrast10"):
        ctx.wbp_filter(torch.from_numpy(img).cuda(), out, -3.5, method)
        X = O.wbp_weight(np.fft.rfft2(mirror_square(img.astype(np.float64), N)), -3.5, A._abi.WBP_METHODS[method],
                         dtype=np.float64)
        expect = np.fft.irfft2(X, s=(N, N))[(N - H) // 2:(N - H) // 2 + H, (N - W) // 2:(N - W) // 2 + W]
        assert rel_l2(out.cpu().numpy(), expect) <= 1e-6, method


@pytest.mark.parametrize("W,H", [(128, 127), (256, 50), (512, 512), (1024, 700)])
def test_slab_stacks_equal_single_slabs(ctx, W, H):
    """The driver's batched slabs (summed forward, fanned backward) against one filter call per slab."""
    print(f"slab stack {W} x {H}", flush=True)
    dims = (40, 40, 12)
    vg = A.volume_geometry(*dims)
    acq = A.Acquisition.build(vg, W, H, [-20.0, 35.0], psis_deg=[2.0, -1.0], shifts=[(0.5, 1.0), (-1.5, 0.0)])
    tdef = [A.TiltDefocus(3000.0, 3150.0, 20.0, -20.0), A.TiltDefocus(2700.0, 2800.0, -50.0, 35.0)]
    ctf = A.ctf_params(pixelsize_nm=0.5, slice_thickness_nm=3.1, beta_fac=(2.0, 0.0, 0.008, 0.0), amp_contrast=0.07)
    sp = A.sart_params(lambda_=0.3, oversampling=2, cut_length=(1, 1), dim_length=(2, 2))
    projs = torch.from_numpy(np.stack([white(H, W, 3), white(H, W, 4)])).cuda()
    vol = torch.zeros(dims[::-1], device="cuda")
    ctx.sart_ctf_run(vg, acq, tdef, projs, vol, sp, ctf, iterations=2)
    ref = torch.zeros_like(vol)
    per_slab_sart_ctf(ctx, vg, acq, tdef, projs, ref, sp, ctf, iterations=2)
    assert float(ref.abs().max()) > 0
    assert torch.equal(vol, ref)


PREP = {
    "uint16_none": dict(dtype="uint16", normalization="none", lp=30.0, lps=6.0),
    "float_std_hp": dict(dtype="float32", normalization="std", lp=0.0, lps=0.0, hp=4.0, hps=2.0),
    "int16_mean_flip_dose": dict(dtype="int16", normalization="mean", mirror_y=True, lp=25.0, lps=5.0,
                                 dose_weighting=True, pixelsize_nm=0.25),
    "int32_wbp_std": dict(dtype="int32", normalization="std", wbp=True, wbp_method="exact", mirror_y=True, lp=35.0,
                          lps=5.0),
    "uint32_wbp_none_raw": dict(dtype="uint32", normalization="none", wbp=True, wbp_method="ramp", skip_filter=True,
                                correct_bad_pixels=False),
}


@pytest.mark.parametrize("W,H", [(128, 90), (101, 256), (512, 512)])
@pytest.mark.parametrize("name", list(PREP))
def test_prepare(ctx, name, W, H):
    """Gates as tests/test_gpu_prep.py's: images and statistics within 1e-5, equal bad-pixel counts; more
    images than one chunk takes leave each image as it is alone."""
    print(f"prepare {name} {W} x {H}", flush=True)
    kw, n = PREP[name], 34
    rng = np.random.default_rng(5)
    yy, xx = np.mgrid[0:H, 0:W]
    imgs = np.rint(800.0 + 100.0 * np.sin(xx / 9.0) - 60.0 * np.cos(yy / 7.0) + rng.normal(0.0, 25.0, (n, H, W)))
    imgs[:, H // 3, 1] = 30000.0
    imgs = imgs.astype(kw["dtype"])
    doses = np.linspace(0.05, 2.0, n).astype(np.float32)
    psis = np.linspace(-4.0, 3.0, n).astype(np.float32)
    pp = A.prep_params(**kw)
    d_in, out = torch.from_numpy(imgs).cuda(), torch.zeros((n, H, W), device="cuda")
    mean, std, bad = ctx.prepare_projections(pp, d_in, out, psi_deg=psis, dose=doses)
    for i in (0, 31, 33):
        ref, m, s, b = P.prepare(imgs[i], psi=float(psis[i]), dose=float(doses[i]),
                                 **{k: v for k, v in kw.items() if k != "dtype"})
        assert b == bad[i]
        assert mean[i] == pytest.approx(m, rel=1e-5, abs=1e-6) and std[i] == pytest.approx(s, rel=1e-5, abs=1e-6)
        assert rel_l2(out[i].cpu().numpy(), ref) < 1e-5
        one = torch.zeros((1, H, W), device="cuda")
        m1, s1, b1 = ctx.prepare_projections(pp, d_in[i:i + 1].contiguous(), one, psi_deg=psis[i:i + 1],
                                             dose=doses[i:i + 1])
        assert torch.equal(one[0], out[i]) and (m1[0], s1[0], b1[0]) == (mean[i], std[i], bad[i])


@pytest.mark.parametrize("W,H", [(256, 256), (1024, 777), (600, 2048)])
def test_subvolume_plan_filters_the_rows_it_reads(ctx, W, H):
    """A CTF plan transforms only the rows of the slab images that its sub-volumes read: the same voxels as
    one whole-image filter per slab, for cubes inside, across and beyond the detector's edges."""
    print(f"sub-volume rows {W} x {H}", flush=True)
    full = A.volume_geometry(W - W % 4, H, 96)
    tilts, rng = [-50.0, 0.0, 33.0], np.random.default_rng(7)
    ctf = A.ctf_params(pixelsize_nm=0.5, slice_thickness_nm=9.3, beta_fac=(2.0, 0.0, 0.008, 0.0), amp_contrast=0.07)
    base = [A.tilt_geometry(t, W, H, psi_deg=4.0, shift=(1.0, -2.0)) for t in tilts]
    kw = dict(ctf=ctf, slab_ranges=[A.defocus_distances(full, g) for g in base],
              defocus=[A.TiltDefocus(3000.0, 3200.0, 15.0, t) for t in tilts])
    geo, geoms = [], []
    for n, x, y, z in ((16, 0.5, 0.5, 0.5), (32, 0.2, 0.9, 0.4), (24, 0.0, 0.02, 0.6), (16, 0.7, 1.0, 0.1), (8, 1.2, 1.3, 0.5)):
        geo.append(A.subvolume_geometry(n, 1.0, (1.0, 1.0, 1.0), full, (x * W + 1.0, y * H + 1.0, z * 96 + 1.0)))
        geoms.append([A.subvolume_tilt_geometry(t, W, H, psi_deg=4.0, shift=(1.0, -2.0),
                                                extra_shift=rng.uniform(-2.0, 2.0, 2)) for t in tilts])
    active = np.ones((len(geo), len(tilts)), bool)
    active[0, 1] = False
    images = torch.from_numpy(np.stack([white(H, W, i) for i in range(len(tilts))])).cuda()
    sets = [[(g, torch.zeros((g.nz, g.ny, g.nx), device="cuda")) for g in geo] for _ in range(2)]
    A.subvol_wbp_plain(ctx, sets[0], geoms, images, 2, active=active, **kw)
    plan = A.SubvolPlan(ctx, sets[1], geoms, images, 2, active=active, tuning=A.SubvolTuning(0, 0, 1, 2), **kw)
    plan.execute()
    torch.cuda.synchronize()
    plan.close()
    assert float(sets[0][0][1].abs().max()) > 0   # (some of the others miss a narrow detector)
    for (_, a), (_, b) in zip(*sets):
        assert torch.equal(a, b)


# At a pixel of 0.5 nm the envelope's exponent is 100 beta_fac[2] at the edge of an axis: 5, and three steep ones
# whose exp underflows before the corner (twice as much), before the edge and well within it; a negative one
# (growing), odd powers, and phase flips (no envelope).
ENVELOPES = {
    "mild": dict(beta_fac=(2.0, 0.0, 0.05, 0.0)),
    "exponent_800": dict(beta_fac=(2.0, 0.0, 8.0, 0.0)),
    "exponent_1500": dict(beta_fac=(2.0, 0.0, 15.0, 0.0)),
    "exponent_3000": dict(beta_fac=(0.0, 0.0, 30.0, 0.0)),
    "growing": dict(beta_fac=(2.0, 0.0, -0.05, 0.0)),
    "odd_powers": dict(beta_fac=(2.0, 0.3, 0.008, 0.01)),
    "phase_flip": dict(beta_fac=(2.0, 0.0, 0.008, 0.0), phase_flip_only=True),
}


@pytest.mark.parametrize("W,H", [(128, 128), (256, 131), (512, 512), (1000, 1024)])
@pytest.mark.parametrize("name", list(ENVELOPES))
def test_slab_filter_envelopes(ctx, name, W, H):
    """Every form of the CTF's envelope, against the FP64 composition: a factor scales a point's rounding error
    with its value, so the gate is that of white images (above)."""
    print(f"envelope {name} {W} x {H}", flush=True)
    kw = ENVELOPES[name]
    img = white(H, W, W + H)
    corners, cut, dim = [0, H - 1, W - 1, H - 1, 0, 0, W - 1, 0], (0.0, 0.0), (2.0, 2.0)
    p = A.ctf_params(pixelsize_nm=0.5, amp_contrast=0.07, **kw)
    k = O.ctf_consts(2.7, 300.0, 0.5, max(W, H), 0.07)
    for for_fp in (True, False):
        out = torch.zeros((H, W), device="cuda")
        ctx.ctf_slab_filter(torch.from_numpy(img).cuda(), out, corners, p, 3000.0, 3150.0, 20.0, for_fp=for_fp,
                            accumulate=False, cut_length=cut, dim_length=dim)
        _, f = CC.slab_filter(img.astype(np.float64), corners, k, 3000.0, 3150.0, 20.0, for_fp, cut, dim,
                              beta=kw["beta_fac"], phase_flip=kw.get("phase_flip_only", False))
        assert float(np.abs(f).max()) > 0
        assert rel_l2(out.cpu().numpy(), f) <= 1e-6, for_fp


def test_ctf_factor_near_its_zeros(ctx):
    """The factor itself where it is small, so that an absolute error of the phase's sine and cosine shows beside
    the float rounding: sine and cosine of equal weight put the zeros an eighth of a turn off, where truncated
    polynomials err most.  Phases to 40 radians carry 40 * 2^-53 * 4 operations = 2e-14 in either arithmetic, and
    without damping the factor's slope at a zero is 1 / wiener = 10: 4e-13, gate 2e-12 beside the rounding.
    (Column 0 is left out: there the oracle's angle is the float pi / 2.)"""
    N = 1024
    print(f"factor near zeros {N}", flush=True)
    beta = (0.0, 0.0, 0.0, 0.0)
    p = A.ctf_params(pixelsize_nm=0.5, amp_contrast=0.70710678, beta_fac=beta)
    k = O.ctf_consts(2.7, 300.0, 0.5, N, 0.70710678)
    ones = np.ones((N, N // 2 + 1), np.complex64)
    spec = torch.from_numpy(ones).cuda()
    ctx.ctf_apply(spec, p, 3000.0, 3150.0, 20.0, for_fp=False)
    got = spec.cpu().numpy().real[:, 1:].astype(np.float64)
    ref = O.ctf_apply(ones.astype(np.complex128), k, 3000.0, 3150.0, 20.0, for_fp=False, beta=beta).real[:, 1:]
    assert float(np.abs(ref).min()) < 4e-5   # zeros are met (3.2e-5)
    assert np.all(np.abs(got - ref) <= 2.0 ** -23 * np.abs(ref) + 2e-12)


@pytest.mark.parametrize("N", [128, 512, 2048])
def test_prepared_squares_have_no_mean(ctx, N):
    """A square whose mean is 30000 times its deviation: the normalised image has none of it left.  Without
    frequency 0 a pixel's error is a few 2^-24 of the deviation 1, independent of the others' or a bias of that
    size: gate 1e-6.  (Subtracted from pixels of its size, 2^-9 apart, it left their rounding in the deviation.)"""
    print(f"mean of a prepared square {N}", flush=True)
    img = (30000.3 + white(N, N, 11)).astype(np.float32)
    out = torch.zeros((1, N, N), device="cuda")
    pp = A.prep_params(dtype="float32", normalization="std", lp=0.4 * N, lps=0.05 * N)
    mean, std, _ = ctx.prepare_projections(pp, torch.from_numpy(img[None]).cuda(), out)
    assert mean[0] == pytest.approx(float(img.astype(np.float64).mean()), rel=1e-6)
    got = out[0].double()
    assert abs(float(got.mean())) <= 1e-6
    assert float(got.std(unbiased=False)) == pytest.approx(1.0, rel=1e-5)


def test_filters_take_the_memory_they_use(gpu):
    """A context holds one spectrum (2048: 17 MB) and the crop weights (17 MB) for single images, and 33 spectra
    (555 MB) for a stack that is prepared; the slab images (537 MB) are the summed slabs' alone."""
    N = 2048
    print(f"filter memory {N}", flush=True)
    p = A.ctf_params(pixelsize_nm=0.5)
    pp = A.prep_params(dtype="float32", normalization="std", lp=0.4 * N, lps=0.05 * N)

    def used(c, n, what):
        img, out = torch.ones((2, n, n), device="cuda"), torch.zeros((2, n, n), device="cuda")
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        if what == "wbp":
            c.wbp_filter(img[0], out[0], 1.0)
        elif what == "slab":
            c.ctf_slab_filter(img[0], out[0], [0, n - 1, n - 1, n - 1, 0, 0, n - 1, 0], p, 3000.0, 3100.0, 0.0,
                              dim_length=(2.0, 2.0))
        else:
            c.prepare_projections(pp, img, out)
        torch.cuda.synchronize()
        return before - torch.cuda.mem_get_info()[0]

    for what, gate in (("wbp", 48), ("slab", 64), ("prepare", 640)):
        c = A.ArtiaContext(0)
        used(c, 128, what)   # kernels loaded
        took = used(c, N, what)
        c.close()
        assert took <= gate << 20, (what, took >> 20)


def test_single_image_filters_in_a_captured_graph(gpu):
    """After one single-image filter the others of its size allocate nothing: captured, and replayed with new images
    between eager calls, they give the eager results."""
    N = 256
    print(f"captured filters {N}", flush=True)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = A.ArtiaContext(0)
    p, corners = A.ctf_params(pixelsize_nm=0.5), [0, N - 1, N - 1, N - 1, 0, 0, N - 1, 0]
    img, work, out = (torch.zeros((N, N), device="cuda") for _ in range(3))

    def filters(dst):
        work.copy_(img)
        c.wbp_filter(work, dst, 1.0, "ramp")
        c.ctf_slab_filter(work, dst, corners, p, 3000.0, 3100.0, 0.0, accumulate=True, dim_length=(2.0, 2.0))

    with torch.cuda.stream(stream):
        c.wbp_filter(work, out, 1.0, "ramp")
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            filters(out)
        for seed in range(4):
            img.copy_(torch.from_numpy(white(N, N, seed)).cuda())
            eager = torch.zeros_like(out)
            filters(eager)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert float(eager.abs().max()) > 0
            assert torch.equal(out, eager)
    c.close()
