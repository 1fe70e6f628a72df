"""Which node-to-lane map a lattice takes (hybird_amd/csrc/lattice.h), on the host: every launch must hold less than
2^32 lanes along x, and enough for the lattice."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SRC = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "lattice.h"
using namespace hyb;
int main() {
    int X, Y, Z;
    while (std::scanf("%d %d %d", &X, &Y, &Z) == 3)
        for (Prec prec : {Prec::F64, Prec::F32S}) {
            LBKParams p{};
            p.X = X; p.Y = Y; p.Z = Z;
            const bool merge = merge_map(p, prec);
            const dim3 g = merge ? merge_grid(p) : row_grid(p), b = row_block(p);
            std::printf("%d %u %u %u %u\n", merge ? 1 : 0, g.x, g.y, g.z, b.x);
        }
    return 0;
}
"""

SIZES = [(3, 17, 19), (40, 150, 150), (256, 256, 256), (257, 150, 150), (3, 8191, 8192), (3, 8192, 8192), (3, 8300, 8300),
         (13, 11000, 12000), (25, 8700, 8000), (64, 5000, 4500), (65, 5000, 4500), (129, 4000, 3000)]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_launches_hold_the_lattice(tmp_path):
    src, exe = tmp_path / "maps.hip", tmp_path / "maps"
    src.write_text(SRC)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-w", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "hybird_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe)], check=True, stderr=subprocess.DEVNULL)
    r = subprocess.run([str(exe)], input="\n".join("%d %d %d" % s for s in SIZES), capture_output=True, text=True,
                       check=True)
    rows = [tuple(int(v) for v in l.split()) for l in r.stdout.splitlines()]
    assert len(rows) == 2 * len(SIZES)
    merged = 0
    for k, (merge, gx, gy, gz, lanes) in enumerate(rows):
        X, Y, Z = SIZES[k // 2]
        assert gx * lanes < 2 ** 32, (SIZES[k // 2], merge)
        waves = -(-X // 64)  # wavefronts of a row
        assert gx * gy * gz * (lanes // 64) >= waves * Y * Z, (SIZES[k // 2], merge)
        merged += merge
    assert 0 < merged < len(rows)
