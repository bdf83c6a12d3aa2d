"""The plain form's own sine and cosine (sincos_near): the error of its
polynomials, and how often and how far its results are off the correctly rounded
ones, for the function itself compiled for the host (CPU)."""
import os
import re
import subprocess

import numpy as np
import pytest

from conftest import ROOT

HEADER = os.path.join(ROOT, "gpu_lomb_scargle_amd", "csrc", "ls_device.h")
NUM = r"-?0x1(?:\.[0-9a-f]+)?p[+-]\d+"


def _source():
    text = open(HEADER).read()
    a = text.index("constexpr double kTrigFar")
    return text[a:text.index("\n}\n", a) + 3]


def _polynomials():
    """(sine, cosine) coefficients, highest power first, of the two variants; the
    last coefficient of the carried ones is a sum of two doubles."""
    body = _source()
    carried, short = body[body.index("if constexpr (CARRIED)"):].split("} else {", 1)
    get = lambda part, name: [[float.fromhex(c)] for line in re.findall(r"(?:double )?" + name + r" = fma\(.*", part)
                              for c in re.findall(NUM, line)]
    out = []
    for part, ks in ((carried, ("kS", "kC")), (short, (None, None))):
        for name, k in zip("pq", ks):
            c = get(part, name)
            if k:
                c[-1].append(float.fromhex(re.search("const double " + k + " = (" + NUM + ")", part).group(1)))
            out.append(c)
    return out


def test_error_of_the_polynomials():
    """|sin h - (h + h^3 p(h^2))| and |cos h - (1 - h^2/2 + h^4 q(h^2))| on
    |h| <= pi/4, in units of 2^-53: far below the rounding of the results."""
    mp = pytest.importorskip("mpmath")
    mp.mp.dps = 50
    bounds = [0.001, 0.001, 0.08, 0.02]  # carried sine and cosine, the others
    degrees = [6, 6, 5, 5]
    for c, first, bound, degree, odd in zip(_polynomials(), (3, 4) * 2, bounds, degrees, (1, 0) * 2):
        c = [sum(mp.mpf(v) for v in part) for part in c]
        assert len(c) == degree + 1
        worst = 0
        for i in range(1, 601):
            h = mp.pi / 4 * i / 600
            exact = mp.sin(h) - h if odd else mp.cos(h) - 1 + h * h / 2
            worst = max(worst, abs(mp.polyval(c, h * h) * h ** first - exact))
        assert worst * 2 ** 53 < bound, (first, mp.nstr(worst * 2 ** 53, 4))


PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
using std::fma;
typedef long long ll;
static ll __double_as_longlong(double x) { ll v; std::memcpy(&v, &x, 8); return v; }
static double __longlong_as_double(ll v) { double x; std::memcpy(&x, &v, 8); return x; }
%s
template <bool CARRIED> void check(double most) {
    uint64_t r = 88172645463325252ull, off = 0;
    double worst = 0.0;
    const int n = 200000;
    for (int i = 0; i < n; ++i) {
        r ^= r << 13; r ^= r >> 7; r ^= r << 17;
        const double x = ((double)(r >> 11) * 0x1p-53 * 2.0 - 1.0) * most;
        double s, c;
        sincos_near<CARRIED>(x, &s, &c);
        const long double e[2] = {sinl((long double)x), cosl((long double)x)};
        const double g[2] = {s, c};
        for (int q = 0; q < 2; ++q) {
            off += g[q] != (double)e[q];
            int ex;
            (void)std::frexp((double)e[q], &ex);
            const double ulp = std::ldexp(1.0, ex - 53), d = std::fabs((double)((long double)g[q] - e[q])) / ulp;
            if (d > worst) worst = d;
        }
    }
    std::printf("%%d %%g %%.6f %%.4f\n", (int)CARRIED, most, (double)off / (2.0 * n), worst);
}
int main() {
    for (double most : {10.0, 1e3, 2.7e5, 4e8}) { check<false>(most); check<true>(most); }
}
"""


@pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="needs an 80-bit long double to compare with")
def test_results_against_the_correctly_rounded_ones(tmp_path):
    """At most 1.8% (carried 0.1%) of the results are not the correctly rounded
    ones, none by more than 0.75 (0.52) ulp."""
    body = re.sub(r"#pragma clang.*", "", _source()).replace("__device__ __forceinline__ ", "static ")
    src, exe = tmp_path / "trig.cpp", tmp_path / "trig"
    src.write_text(PROGRAM % body)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", str(src), "-o", str(exe)], check=True,
                   capture_output=True, timeout=120)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout.splitlines()
    assert len(lines) == 8
    for line in lines:
        carried, most, share, worst = line.split()
        print(line)
        assert float(share) <= (0.001 if carried == "1" else 0.018), line
        assert float(worst) <= (0.52 if carried == "1" else 0.75), line
