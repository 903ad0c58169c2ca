"""The grid cell of an ion on the PME mesh does not depend on how the compiler
fuses multiplications and additions.  The cell is formed in three kernels, and
a brick's ions reach LDS relative to it, so for ions on the faces of grid cells
a rounding that differs between two of them would name different bricks.  The
header is compiled for the host twice, with the contractions of a device build
and with none, and must give the same cells and offsets bit for bit."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SRC = """
#include "pme_cell.hpp"
#include <cstdio>
int main(int argc, char **argv)
{
    using namespace agpu;
    int h[4];
    CellArg B;
    PmeGrid g{};
    FILE *in = fopen(argv[1], "rb"), *out = fopen(argv[2], "wb");
    if (fread(h, 4, 4, in) != 4 || fread(B.A, 8, 9, in) != 9) return 1;
    for (int d = 0; d < 3; ++d) g.K[d] = h[1 + d];
    for (int n = 0; n < h[0]; ++n) {
        double r[3];
        if (fread(r, 8, 3, in) != 3) return 1;
        for (int e = 0; e < 3; ++e) {
            int ib;
            const double v[2] = {pme_cell(B, g, e, r[0], r[1], r[2], ib), 0.0};
            const double w[2] = {v[0], (double)ib};
            fwrite(w, 8, 2, out);
        }
    }
    return fclose(out);
}
"""


def face_ions(cell, K, rng, n):
    """Ions on faces of grid cells (every eighth one a face of a brick) and
    one ulp of a coordinate to either side, in and around the cell."""
    frac = (rng.integers(0, 1 + np.array(K) // 8, (n, 3)) * 8.0 / np.array(K)) - 0.5 + rng.integers(-2, 3, (n, 3))
    free = rng.random((n, 3)) < 0.3
    frac = np.where(free, rng.random((n, 3)), frac)
    r = frac @ cell
    for step in (-np.inf, np.inf):
        k = rng.random(r.shape) < 0.25
        r = np.where(k, np.nextafter(r, step), r)
    return r


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("K", [(8, 16, 24), (40, 41, 64), (160, 160, 160)])
def test_cell_does_not_depend_on_contraction(tmp_path, K):
    src = tmp_path / "cell.hip"
    src.write_text(SRC)
    rng = np.random.default_rng(K[1])
    cell = np.diag([9.1, 10.3, 12.7]) @ (np.eye(3) + 0.15 * np.array([[0, 1, 0.5], [1, 0, -0.4], [0.5, -0.4, 0]]))
    r = face_ions(cell, K, rng, 20000)
    arg = tmp_path / "in"
    with open(arg, "wb") as f:
        np.array([len(r), *K], np.int32).tofile(f)
        np.linalg.inv(cell).T.astype(np.float64).reshape(-1).tofile(f)
        r.tofile(f)
    res = []
    for mode in ("off", "fast-honor-pragmas"):
        exe = tmp_path / ("cell_" + mode)
        subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-host-only", "-mfma", "-ffp-contract=" + mode,
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "atomistica_amd", "csrc"),
                        str(src), "-o", str(exe)], check=True, capture_output=True)
        out = tmp_path / ("out_" + mode)
        subprocess.run([str(exe), str(arg), str(out)], check=True)
        res.append(np.fromfile(out).reshape(-1, 3, 2))
    a, b = res
    assert np.all((a[..., 1] >= 0) & (a[..., 1] < np.array(K)))
    assert np.array_equal(a[..., 1], b[..., 1]), "cells differ"
    assert np.array_equal(a[..., 0], b[..., 0]), "offsets differ"
