"""LDS arrays of the sweep kernels against the indices that reach them (CPU)."""
import glob
import os
import re

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
