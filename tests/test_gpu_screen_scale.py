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
