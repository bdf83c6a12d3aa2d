"""The plain form on both sides of the phase where its sine and cosine change
hands (omega t = 2^30, decided per 256 staged observations): phases below it,
above it, and both in one block and across blocks, against the CPU oracle.

Tolerances: the plain form's own, 1e-12 for the FP64 standard variant (tests/
test_gpu_parity.py).  Generalized FP64: the reference's second pass rounds
t - tau to 9e-10 d at t ~ 7e6 d, 1.4e-7 rad; a last-bit difference of tau moves
that rounding in ~1e-9 of the terms, so 1e-9 on bins of at least 1e-3 Pmax.
FP32 against the oracle with correctly rounded float libm: 1e-5 on bins of at
least 1e-2 Pmax.
"""
import numpy as np
import pytest

import oracle
from gpu_lomb_scargle_amd import _native, synth
from test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu
EDGE = 2.0 ** 30 / synth.OMEGA_MAX  # days


@pytest.mark.parametrize("gen", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [40, 256, 257, 600])
def test_phase_range(n, dtype, gen):
    rng = np.random.default_rng(n)
    ts, ys, ds = [], [], []
    for lo, hi in ((0.0, 400.0), (0.3 * EDGE, 0.9 * EDGE), (0.9 * EDGE, 1.3 * EDGE), (1.4 * EDGE, 3.0 * EDGE)):
        t = np.sort(rng.uniform(lo, hi, n)).astype(dtype)
        ts.append(t)
        ys.append((np.sin(3.1 * t.astype(np.float64)) + rng.normal(0, 0.3, n)).astype(dtype))
        ds.append(np.exp(rng.uniform(np.log(0.01), np.log(0.2), n)).astype(dtype))
    o = np.repeat(np.arange(4, dtype=np.uint32), n)
    t, y, dy = np.concatenate(ts), np.concatenate(ys), np.concatenate(ds) if gen else None
    nf = 1009
    r = _native.batch_host(o, t, y, dy, synth.OMEGA_MIN, synth.OMEGA_MAX, nf,
                           _native.GENERALIZED if gen else _native.STANDARD, dtype, _native.FORM_PLAIN)
    with oracle.float_libm_cr():
        ref = oracle.batch(o, t, y.copy(), dy, synth.OMEGA_MIN, synth.OMEGA_MAX, nf, gen, dtype, nthreads=8)[0]
    if dtype == np.float32:
        assert_close(r["pgram"], ref, 1e-5, 1e-2, 1e-5)
    elif gen:
        assert_close(r["pgram"], ref, 1e-9, 1e-3, 1e-9)
    else:
        assert_close(r["pgram"], ref, 1e-12, 1e-6, 1e-12)
