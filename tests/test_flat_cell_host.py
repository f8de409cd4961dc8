"""The flat walk's cell sum (flat_walk.hpp), compiled for the host, on cells whose terms before the last
rounding are exact: edges that are integers below 2^10 and middles in 64ths take at most 22 bits.  What is
left are the sum's own rounding, 2^-24 of it, and two in the second-moment term h, 2^-23 of it."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np

from artiatomi_amd import build as B

SRC = """
#include "artia_internal.hpp"
#include "flat_walk.hpp"
extern "C" void cell_sums(const float* in, int n, float* out) {
    for (int i = 0; i < n; i++, in += 8)
        out[i] = artia::flat_cell_sum(in[0], in[1], in[2], in[3], in[4], in[5], in[6], in[7]);
}
"""


def test_flat_cell_sum_is_rounded_once(tmp_path):
    src, lib = tmp_path / "cell.hip", tmp_path / "cell.so"
    src.write_text(SRC)
    root = Path(B.PKG).parent
    subprocess.run([B.hipcc(), "--offload-host-only", "-mfma", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                    "-I", str(B.CSRC), "-I", str(root / "include"), "-o", str(lib), str(src)], check=True)
    rng, n = np.random.default_rng(1), 200000
    cells = np.empty((n, 8), np.float32)
    cells[:, :4] = rng.integers(0, 1024, (n, 4))
    cells[:, 4:6] = rng.integers(0, 65, (n, 2)) / 64.0
    cells[:, 6] = rng.integers(0, 12, n)
    cells[:, 7] = rng.uniform(0.0, 2e-5, n)
    out = np.empty(n, np.float32)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    C.CDLL(str(lib)).cell_sums(ptr(cells), n, ptr(out))
    A_, B_, C_, D_, a, c, m, K = cells.astype(np.float64).T
    e0, e1 = A_ + a * (B_ - A_), C_ + a * (D_ - C_)
    h = (D_ - C_ - B_ + A_) * K * m * (m * m - 1.0)
    ref = m * (e0 + c * (e1 - e0)) + h
    assert np.all(out[m == 0] == 0.0)
    assert np.all(np.abs(out - ref) <= 2.0 ** -24 * np.abs(ref) + 2.0 ** -23 * np.abs(h))
