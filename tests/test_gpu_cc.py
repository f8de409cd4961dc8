"""The shift search's tiled correlation over window sizes around its tiles (80 columns; rows by slices) and
shifts around its runs of 9 columns, against the FP64 oracle (oracle/cc_search.py) on white windows.

Tolerance: the map is a double correlation rounded to float, at most 1 in magnitude: 2^-25 rounding and
about 1e-12 of summation order; gate 1e-7.  Peaks are equal (white noise has no ties).
"""
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

import artiatomi_amd as A

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import cc_search  # noqa: E402

pytestmark = pytest.mark.gpu

WINDOWS = [(1, 1), (8, 33), (79, 7), (80, 80), (81, 64), (161, 20), (33, 150)]


@pytest.fixture(scope="module")
def ctx(gpu):
    c = A.ArtiaContext(0)
    yield c
    c.close()


@pytest.mark.parametrize("max_shift", [0, 1, 4, 9, 12, 13, 22, 32])
def test_tiled_correlation(ctx, max_shift):
    print(f"cc max shift {max_shift}", flush=True)
    W = 256
    full = A.volume_geometry(64, 64, 24)
    vg = A.subvolume_geometry(16, 1.0, (1.0, 1.0, 1.0), full, (32.0, 32.0, 12.0))
    g = A.tilt_geometry(20.0, W, W)
    pairs = [(0, 40, 44, w, h) for w, h in WINDOWS]
    ps = A.PairSet(ctx, [(vg, 0)], pairs, [g] * len(pairs))
    try:
        rng = np.random.default_rng(max_shift)
        m, t = (rng.standard_normal(ps.n_pixels).astype(np.float32) for _ in range(2))
        for multi in (False, True):
            peak, cc, ccmap = ps.cc_search(torch.from_numpy(m).cuda(), torch.from_numpy(t).cuda(), W, max_shift,
                                           want_map=True, multi_peak=multi)
            peak, cc, ccmap = peak.cpu().numpy(), cc.cpu().numpy(), ccmap.cpu().numpy()
            for p, (_, x0, y0, w, h) in enumerate(pairs):
                off = ps.windows[p][5]
                a, b = (cc_search.to_square(v[off:off + w * h].reshape(h, w).astype(np.float64), W, x0, y0)
                        for v in (t, m))
                rx, ry, _, ref = cc_search.get_displacement(a, b, max_shift, multi_peak=multi)
                # (a single pixel overlaps itself at no shift only: all others tie, but for the oracle's rounding)
                assert w * h == 1 or (peak[p, 0], peak[p, 1]) == (rx, ry), (w, h)
                cref = cc_search.cc_map_of(ref, max_shift)
                r = np.arange(-max_shift, max_shift + 1)
                # (where every shift anti-correlates the search fails with the disk's maximum as its value)
                assert abs(cc[p] - cref[np.hypot(r[:, None], r) <= max_shift].max()) <= 1e-7
                assert np.abs(ccmap[p] - cref).max() <= 1e-7
    finally:
        ps.close()
