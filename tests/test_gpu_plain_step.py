"""The plain standard FP64 sweep whose bins are stepped from one another, where
it can go wrong: observation counts around the staged block and around the
least count it takes, ragged chunks, grids that start at, below and above its
step or cross zero, phases past its range, identical and NaN times.

Against the CPU oracle at the plain form's 1e-12 (tests/test_gpu_parity.py),
and against the sweep with a sine and cosine per bin, chosen by its tile: what
the stepped sweep leaves to the direct sums is the same arithmetic, so those
bins are equal bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_lomb_scargle_amd import _native, synth
from test_gpu_parity import F64, assert_close

pytestmark = pytest.mark.gpu
COUNTS = [5, 15, 16, 17, 64, 255, 256, 257, 700]
NF = 40013  # times 9 objects: enough bins for the stepped sweep with 8 bins per thread


def _curves(counts, span=1800.0, t0=0.0):
    rng = np.random.default_rng(5)
    ts = [t0 + np.sort(rng.integers(0, int(span), n) + rng.uniform(0, 0.3, n)) for n in counts]
    ys = [np.sin(3.1 * t) + rng.normal(0, 0.3, len(t)) for t in ts]
    return np.repeat(np.arange(len(counts), dtype=np.uint32), counts), np.concatenate(ts), np.concatenate(ys)


def _sweep(o, t, y, lo, hi, tile=None, nf=NF, **kw):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    p = device.SweepPlan(*device.numpy_to_device(o, t, y, None, F64), min_freq=lo, max_freq=hi, num_freqs=nf,
                         variant=_native.STANDARD, form=_native.FORM_PLAIN, top_k=3, tile=tile, **kw)
    p.run()
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in p.results().items()}


@pytest.mark.parametrize("nf", [NF, 300007])  # 8 and 16 bins per thread
@pytest.mark.parametrize("schedule", [_native.SCHEDULE_GRID, _native.SCHEDULE_PERSISTENT])
@pytest.mark.parametrize("t0", [0.0, 51075.0, 2458652.0])
def test_against_the_oracle(t0, schedule, nf):
    o, t, y = _curves(COUNTS, t0=t0)
    r = _sweep(o, t, y, synth.OMEGA_MIN, synth.OMEGA_MAX, nf=nf, schedule=schedule)
    ref = oracle.batch(o, t, y.copy(), None, synth.OMEGA_MIN, synth.OMEGA_MAX, nf, False, F64, nthreads=8)[0]
    assert_close(r["pgram"], ref, 1e-12, 1e-6, 1e-12)
    for k in range(len(COUNTS)):
        best = np.lexsort((np.arange(nf), -r["pgram"][k]))[:3]
        assert np.array_equal(r["index"][k], best) and np.array_equal(r["power"][k], r["pgram"][k][best])


@pytest.mark.parametrize("lo,hi", [(0.0, 60.0), (1e-4, 60.0), (0.09, 60.0), (0.1, 60.0), (-20.0, 40.0), (-60.0, -1.0)])
def test_grids_near_zero(lo, hi):
    """Frequencies below the step have the direct sums' bits (0/0 at frequency 0
    included), all others are within 1e-12."""
    o, t, y = _curves(COUNTS)
    a, b = (_sweep(o, t, y, lo, hi, tile)["pgram"] for tile in (None, (256, 2)))
    om = lo + (hi - lo) / NF * np.arange(NF)
    low = np.abs(om) < 0.999 * 64 * (hi - lo) / NF
    assert np.array_equal(a[:, low], b[:, low], equal_nan=True)
    small = np.array(COUNTS) < 16
    assert np.array_equal(a[small], b[small], equal_nan=True)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert_close(a, b, 1e-12, 1e-6, 1e-12)


def test_phases_past_the_range_and_odd_times():
    """One observation past 2^28 rad, all times equal, and a NaN time: the whole
    object (or the chunks that reach it) has the direct sums' bits."""
    o, t, y = _curves([300, 300, 300, 300])
    t[250] = 2.0 ** 28 / synth.OMEGA_MIN * 1.01
    t[300:600] = 3.5
    t[700] = np.nan
    y[300:600] -= y[300:600].mean()
    # two copies of each: enough bins for the stepped sweep
    o, t, y = np.concatenate([o + 4 * k for k in range(2)]), np.tile(t, 2), np.tile(y, 2)
    a, b = (_sweep(o, t, y, synth.OMEGA_MIN, synth.OMEGA_MAX, tile)["pgram"] for tile in (None, (256, 2)))
    for k in (0, 1, 2, 4, 5, 6):
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    assert_close(a[3], b[3], 1e-12, 1e-6, 1e-12)
    assert np.array_equal(a[3], a[7])


def test_parts_of_a_host_call(monkeypatch):
    """A host call swept in parts (budget of 3 objects, slices of 2; the last
    part alone would be small) has the bits of the call swept whole."""
    o, t, y = _curves([90] * 8)
    args = (o, t, y, None, 1.0, 60.0, 20011, _native.STANDARD, F64, _native.FORM_PLAIN)
    whole = _native.batch_host(*args)
    monkeypatch.setenv("LSAMD_PGRAM_BUDGET_BYTES", str(3 * 20011 * 8))
    monkeypatch.setenv("LSAMD_SLICE_BYTES", str(2 * 20011 * 8))
    parts = _native.batch_host(*args)
    assert np.array_equal(whole["pgram"], parts["pgram"]) and np.array_equal(whole["index"], parts["index"])


@pytest.mark.parametrize("t0,lo,hi", [(0.0, synth.OMEGA_MIN, synth.OMEGA_MAX), (51075.0, 0.63, 62.8), (0.0, 0.3, 60.0),
                                      (0.0, -60.0, -1.0)])
def test_generalized_against_the_oracle(t0, lo, hi):
    """The second pass of the generalized sweep, stepped from 32 observations on,
    around the staged blocks.  A last-bit difference of tau moves the rounding of
    t - tau (test_gpu_plain_phase_range.py): 1e-9 on bins of at least 1e-3 Pmax."""
    counts = [5, 31, 32, 33, 64, 255, 256, 257, 700]
    o, t, y = _curves(counts, t0=t0)
    dy = np.random.default_rng(6).uniform(0.05, 0.3, len(t))
    r = _native.batch_host(o, t, 17.0 + y, dy, lo, hi, 5003, _native.GENERALIZED, F64, _native.FORM_PLAIN)
    ref = oracle.batch(o, t, 17.0 + y, dy, lo, hi, 5003, True, F64, nthreads=8)[0]
    assert np.array_equal(np.isnan(r["pgram"]), np.isnan(ref))
    assert_close(r["pgram"], ref, 1e-9, 1e-3, 1e-9)


def test_generalized_grid_over_zero():
    """tau is 0/0 at frequency 0: NaN there and nowhere else; a NaN time gives an
    object of NaN.  (5003 bins from -20 to 30, and from 0.)"""
    o, t, y = _curves([40, 300, 300])
    dy = np.random.default_rng(6).uniform(0.05, 0.3, len(t))
    t[400] = np.nan
    for lo, hi in ((0.0, 30.0), (-20.0, 30.02)):
        r = _native.batch_host(o, t, y.copy(), dy, lo, hi, 5003, _native.GENERALIZED, F64, _native.FORM_PLAIN)["pgram"]
        ref = oracle.batch(o, t, y.copy(), dy, lo, hi, 5003, True, F64, nthreads=8)[0]
        assert np.array_equal(np.isnan(r), np.isnan(ref))
        far = np.abs(lo + (hi - lo) / 5003 * np.arange(5003)) > 0.1
        for k in (0, 1):  # (object 2 holds the NaN)
            assert_close(r[k][far], ref[k][far], 1e-9, 1e-3, 1e-9)
