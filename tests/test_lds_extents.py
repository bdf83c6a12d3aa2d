"""LDS arrays of the sweep kernels against the indices that reach them (CPU)."""
import glob
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "gpu_lomb_scargle_amd", "csrc")


def test_a_second_view_of_an_lds_array_is_bounded_by_it():
    """Where a kernel uses a __shared__ array through a pointer of another type,
    a static_assert bounds that use by the array's own size: what lies behind a
    __shared__ array is the compiler's choice."""
    views = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        text = open(path).read()
        for m in re.finditer(r"reinterpret_cast<\s*\w+\s*\*>\((s_\w+)\)", text):
            views += 1
            name = m.group(1)
            assert re.search(r"static_assert\(sizeof\(" + name + r"\) >= ", text[m.end():m.end() + 400]), (path, name)
    assert views > 0


EXTENTS = r"""
#include "ls_interp.h"
#include <cstdio>
using namespace lsamd;
int main() {
    for (int screen = 0; screen < 2; ++screen)
        for (int mode = 1; mode <= kIpModes; ++mode) {
            const unsigned rows = (unsigned)ip_rows(mode), m = (unsigned)ip_per_row(mode);
            unsigned z = 0, x = 0;
            for (unsigned t = 0; 32 * t < rows; ++t)
                for (unsigned l = 0; l < 64; ++l) {
                    const unsigned s = ip_operand_row(rows, t, l & 31), zo = m * s + 8 * (l >> 5), xo = 2 * m * s + 8 * (l >> 5);
                    if (zo + 7 > z) z = zo + 7;
                    const unsigned xe = xo + (ip_wide(screen, mode) ? 16 : 0) + 7;
                    if (xe > x) x = xe;
                }
            std::printf("%d %d %d %u %u %u %u\n", screen, mode, ip_step(mode), z, kIpPoints, x, kIpPoints2);
        }
}
"""


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="hipcc not available")
def test_operand_reads_of_the_coarse_grid_stay_within_the_points(tmp_path):
    """Every lane of every tile of every mode: the last point that its 16-byte
    operand reads take lies within the array of the sum that it reads."""
    src, exe = tmp_path / "extents.hip", tmp_path / "extents"
    src.write_text(EXTENTS)
    subprocess.run(["/opt/rocm/bin/hipcc", "--cuda-host-only", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                    str(src), "-o", str(exe)], check=True, capture_output=True, timeout=300)
    rows = [[int(v) for v in line.split()] for line in subprocess.run([str(exe)], check=True, capture_output=True,
                                                                      text=True).stdout.splitlines()]
    assert len(rows) == 14
    for screen, mode, h, z, nz, x, nx in rows:
        assert z < nz and x < nx, (screen, mode, h, z, nz, x, nx)
