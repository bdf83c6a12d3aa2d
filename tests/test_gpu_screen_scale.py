"""Peaks without a periodogram, where the screen of the coarse grid could run
out of range or precision.  The peaks equal, bit for bit, those of the objects
swept one by one, which takes the direct sums."""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth

pytestmark = pytest.mark.gpu
F32, F64 = np.float32, np.float64
DF = (synth.OMEGA_MAX - synth.OMEGA_MIN) / (2 * np.pi)  # cycles/day of the whole grid


def check(ts, ys, ds, nf, top_k, dtype, lo=synth.OMEGA_MIN, hi=synth.OMEGA_MAX, **kw):
    """All objects in one call against each alone; returns the call's results."""
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    counts = [len(t) for t in ts]
    o = np.repeat(np.arange(len(ts), dtype=np.uint32), counts)
    dy = None if ds is None else np.concatenate(ds)
    tt, yy, dd, off = device.numpy_to_device(o, np.concatenate(ts), np.concatenate(ys), dy, dtype)
    assert sum(counts) * nf >= 1e9 > max(counts) * nf  # the call takes the screen, an object alone does not
    kw = dict(min_freq=lo, max_freq=hi, num_freqs=nf, form=_native.FORM_SPLIT32, top_k=top_k, pgram=False,
              variant=_native.STANDARD if ds is None else _native.GENERALIZED, **kw)
    all_ = device.sweep(tt, yy, dd, off, **kw)
    torch.cuda.synchronize()
    first = np.concatenate([[0], np.cumsum(counts)])
    for k in range(len(ts)):
        a = slice(first[k], first[k + 1])
        one = device.sweep(tt[a], yy[a], None if dd is None else dd[a], torch.tensor([0, counts[k]], device="cuda"),
                           obs_slices=1, **kw)
        torch.cuda.synchronize()
        for name in ("index", "power", "period"):
            assert torch.equal(all_[name][k], one[name][0]), (k, name, all_[name][k], one[name][0])
    return {k: v.cpu().numpy() for k, v in all_.items()}


@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
@pytest.mark.parametrize("n", [63, 64, 127])
@pytest.mark.parametrize("h", [3, 5, 8, 16])
def test_two_epochs(h, n, gen):
    """Observations at both ends of the span alone, where the window's weights
    are largest (9.9), magnitudes just below a power of two and not centred, the
    oversampling just above the screen's least: the sums at frequencies that
    bring both epochs into phase are nearly the largest that there can be.  The
    epochs are a day long, so that those bins are not ill-conditioned (where
    every power is computed again)."""
    nf, K = 500009, 36
    rng = np.random.default_rng(100 * h + n)
    span = nf / DF / (1.3 * h) * 0.9999
    ts, ys, ds = [], [], []
    for k in range(K):
        t = np.concatenate([rng.uniform(0, 1.0, n // 2), span - rng.uniform(0, 1.0, n - n // 2)])
        t.sort()
        t[0], t[-1] = 0.0, span
        ts.append(t)
        ys.append(0.9999 - 1e-4 * (k + 1) * rng.uniform(0, 1, n))
        ds.append(rng.uniform(0.9, 1.0, n))
    check(ts, ys, ds if gen else None, nf, 3, F64)


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("unit", [1e-37, 1e-30, 1e-26, 1e-20, 1.0, 1e15, 1e24, 1e37])
def test_units_of_the_magnitudes(unit, normalize, dtype):
    """Flux densities in any unit, powers with and without their normalisation;
    where FP32 powers are denormal or infinite, the first of the equal ones is
    the peak.  The same objects in units of 1 have their peaks in the same bins
    (FP64: the unit is a power of two, so that only exponents differ)."""
    rng = np.random.default_rng(17)
    nf, K, n = 400009, 40, 90
    two = 2.0 ** np.round(np.log2(unit))
    ts = [np.sort(rng.uniform(0.0, 1500.0, n)) for _ in range(K)]
    ys = [np.sin(2 * np.pi * rng.uniform(0.3, 20.0) * t) + rng.normal(0, 0.3, n) for t in ts]
    ys[3] = np.zeros(n)
    ys[4] = np.full(n, 3.0)
    r = check(ts, [two * y for y in ys], None, nf, 3, dtype, normalize=normalize)
    if dtype == F64:
        ref = check(ts, ys, None, nf, 3, dtype, normalize=normalize)
        assert np.array_equal(r["index"], ref["index"])
        assert (r["index"][5:, 0] > 0).all() and (r["power"][5:, 0] > 0).all()


@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
@pytest.mark.parametrize("n,nf", [(4001, 60011), (20011, 40009), (65003, 12007)])
@pytest.mark.parametrize("top_k", [1, 3])
def test_evenly_sampled_light_curves(n, nf, top_k, gen):
    """Fluxes every half hour around 1, not centred (standard), with signals of
    0, 10^-4 and 10^-3 of that, or a smooth one without noise, searched where the window's and the signal's
    sidelobes are small: peaks of 10^-5 and less of the magnitudes' own power,
    where the screen's rounding shows."""
    rng = np.random.default_rng(n)
    t = 100.0 + np.arange(n) / 48.0
    T = t[-1] - t[0]
    K = max(2, int(np.ceil(1.05e9 / (n * nf))))
    df = 0.97 / (1.3 * 3 * T)
    lo = 2 * np.pi * 20.0
    ts, ys, ds = [], [], []
    for k in range(K):
        amp = (0.0, 1e-4, 1e-3)[k % 3]
        y = 1.0 + amp * np.sin(2 * np.pi * (20.0 + rng.uniform(0.1, 0.9) * nf * df) * t + k) + 1e-4 * rng.normal(0, 1, n)
        if k % 4 == 3:
            y = 1.0 + 0.01 * np.sin(2 * np.pi * 1.3 * t)
        ts.append(t)
        ys.append(y)
        ds.append(np.full(n, 1e-4))
    check(ts, ys, ds if gen else None, nf, top_k, F64, lo=lo, hi=lo + 2 * np.pi * nf * df)
