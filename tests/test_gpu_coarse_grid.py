"""The coarse-grid sweep of split32.  FP32 periodograms on grids finer than an
object's resolution: every mode and its edges against the plain FP64 form on
the same float inputs, and its peaks against its own periodogram.  Tolerance:
the split forms', relative 1e-5 on bins of at least 1e-3 Pmax and 2e-6 Pmax
absolute (tests/test_gpu_parity.py).  Peaks without a periodogram: equal, bit
for bit, to those of the objects swept one by one, which takes the direct sums.
"""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth
from test_gpu_parity import assert_close, first_strict_max

pytestmark = pytest.mark.gpu
F32, F64 = np.float32, np.float64
DF = (synth.OMEGA_MAX - synth.OMEGA_MIN) / (2 * np.pi)  # cycles/day of the whole grid


def light_curves(counts, spans, gen, seed):
    rng = np.random.default_rng(seed)
    ts, ys, ds = [], [], []
    for n, span in zip(counts, spans):
        t = np.sort(rng.uniform(0.0, span, n))
        if n > 1:
            t[0], t[-1] = 0.0, span
        d = np.exp(rng.uniform(np.log(0.01), np.log(0.2), n))
        f = rng.uniform(0.3, 20.0)
        y = np.sin(2 * np.pi * f * t) + rng.normal(0, 0.3, n)
        ts.append(t.astype(F32))
        ys.append(((17 + 0.3 * y) if gen else y).astype(F32))
        ds.append(d.astype(F32))
    o = np.repeat(np.arange(len(counts), dtype=np.uint32), counts)
    return o, np.concatenate(ts), np.concatenate(ys), np.concatenate(ds) if gen else None


def sweep(o, t, y, dy, nf, dtype, form, top_k=3, gen=False):
    return _native.batch_host(o, t.astype(dtype), y.astype(dtype), None if dy is None else dy.astype(dtype),
                              synth.OMEGA_MIN, synth.OMEGA_MAX, nf,
                              _native.GENERALIZED if gen else _native.STANDARD, dtype, form, top_k=top_k)


# calls of several objects through the host entry point take the coarse grid
# from 2^18 bins on; 33 x 8160 and 9 x 32640 are whole workgroups of the
# smallest and the largest mode
@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
@pytest.mark.parametrize("nf", [262144, 262145, 269279, 269280, 269281, 293760, 300007])
def test_modes_and_edges(nf, gen):
    """Spans that put an object just inside and outside of every coarse step
    (oversampling 3.9 ... 60), observation counts around the 16-observation
    blocks, the 64-observation stages and the 256-observation runs."""
    over = np.array([3.8, 4.0, 7.7, 7.9, 9.5, 9.9, 11.6, 12.2, 15.5, 16.2, 19.3, 20.5, 24.5, 31.0, 33.0, 39.5, 60.0])
    counts = [200, 17, 33, 64, 65, 255, 256, 257, 40, 512, 513, 18, 100, 30, 48, 300, 80]
    o, t, y, dy = light_curves(counts, nf / DF / over, gen, nf)
    r = sweep(o, t, y, dy, nf, F32, _native.FORM_SPLIT32, gen=gen)
    ref = sweep(o, t, y, dy, nf, F64, _native.FORM_PLAIN, gen=gen)
    assert_close(r["pgram"], ref["pgram"], 1e-5, 1e-3, 2e-6)
    for k in range(len(counts)):
        row = r["pgram"][k].copy()
        for q in range(3):  # the reference's three scans over the sweep's own periodogram
            i, p = first_strict_max(row)
            assert r["index"][k, q] == i and r["power"][k, q] == p
            row[i] = 0


def test_objects_without_a_span_or_with_nan():
    """Identical times and few observations stay with the direct sums, a NaN
    magnitude stays in its object, constant magnitudes give no peak; the
    other objects' results do not depend on them."""
    counts = [60, 60, 60, 60, 10, 120]
    o, t, y, dy = light_curves(counts, [500.0] * 6, False, 5)
    nf = 262147
    keep = [0, 5]
    pick = np.isin(o, keep)
    alone = sweep(o[pick], t[pick], y[pick], None, nf, F32, _native.FORM_SPLIT32)
    t[60:120] = 7.0
    y[130] = np.nan
    y[180:240] = 0.0
    r = sweep(o, t, y, None, nf, F32, _native.FORM_SPLIT32)
    for i, k in enumerate(keep):
        assert np.array_equal(r["pgram"][k], alone["pgram"][i])
        assert np.array_equal(r["index"][k], alone["index"][i]) and np.array_equal(r["power"][k], alone["power"][i])
    assert np.isnan(r["pgram"][2]).all() and (r["index"][2] == 0).all() and (r["power"][2] == 0).all()
    assert (r["index"][3] == 0).all()
    direct = sweep(o, t, y, None, nf, F64, _native.FORM_SPLIT32)
    assert_close(r["pgram"][4], direct["pgram"][4], 1e-6, 1e-3, 1e-6)


@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
def test_grid_and_persistent_and_graph_agree(gen):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    o, t, y, dy = light_curves([120, 40, 300, 90], [300.0, 900.0, 1200.0, 5000.0], gen, 9)
    tt, yy, dd, off = device.numpy_to_device(o, t, y, dy, F32)
    kw = dict(min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MAX, num_freqs=262501, obs_slices=1, form=_native.FORM_SPLIT32, top_k=3,
              variant=_native.GENERALIZED if gen else _native.STANDARD)
    ref = device.SweepPlan(tt, yy, dd, off, **kw)
    ref.run()
    a = {k: v.clone() for k, v in ref.results().items()}
    plan = device.SweepPlan(tt, yy, dd, off, schedule=_native.SCHEDULE_PERSISTENT, **kw)
    plan.capture_graph(torch.cuda.Stream())
    for _ in range(3):
        for x in (plan.pgram, plan.peak_power, plan.peak_period, plan.peak_index):
            x.fill_(-1)
        torch.cuda.synchronize()
        plan.run()
        torch.cuda.synchronize()
        for k, v in plan.results().items():
            assert torch.equal(v, a[k]), k


@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("nf,top_k", [(420007, 1), (420007, 3), (440640, 3), (1000000, 3)])
def test_peaks_alone_equal_the_direct_sums(nf, top_k, dtype, gen):
    """Every coarse step and its neighbourhood, observation counts around the
    blocks and stages, noise without a peak, a pair of equal peaks, constant
    and NaN magnitudes; persistent and grid schedules."""
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    over = np.array([3.5, 3.95, 5.1, 5.3, 6.4, 6.6, 7.7, 7.9, 10.3, 10.5, 12.9, 13.1, 20.5, 21.0, 33.0, 60.0, 9.0, 9.0, 9.0, 9.0])
    counts = [200, 17, 33, 64, 65, 255, 256, 257, 12, 512, 513, 18, 100, 30, 48, 300, 90, 120, 60, 80]
    o, t, y, dy = light_curves(counts, nf / DF / over, gen, nf + top_k)
    first = np.concatenate([[0], np.cumsum(counts)])
    rng = np.random.default_rng(8)
    part = lambda k: slice(first[k], first[k + 1])
    y[part(16)] = rng.normal(0, 1, 90)                                          # noise
    tk = t[part(17)].astype(F64)
    y[part(17)] = np.sin(2 * np.pi * 5.0 * tk) + np.sin(2 * np.pi * 11.0 * tk)  # two peaks of one height
    y[part(18)] = 3.0
    y[first[19] + 7] = np.nan
    tt, yy, dd, off = device.numpy_to_device(o, t, y, dy, dtype)
    kw = dict(min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MAX, num_freqs=nf, form=_native.FORM_SPLIT32, top_k=top_k,
              variant=_native.GENERALIZED if gen else _native.STANDARD, pgram=False)
    assert int(first[-1]) * nf >= 1e9  # below, the direct sums
    got = []
    for schedule in (_native.SCHEDULE_GRID, _native.SCHEDULE_PERSISTENT):
        plan = device.SweepPlan(tt, yy, dd, off, schedule=schedule, **kw)
        for x in (plan.peak_power, plan.peak_period, plan.peak_index):
            x.fill_(-1)
        plan.run()
        torch.cuda.synchronize()
        got.append({k: v.clone() for k, v in plan.results().items()})
    for k in range(len(counts)):
        a = part(k)
        one = device.SweepPlan(tt[a], yy[a], None if dd is None else dd[a], torch.tensor([0, counts[k]], device="cuda"),
                               obs_slices=1, **kw)
        one.run()
        torch.cuda.synchronize()
        for name, v in one.results().items():
            for g in got:
                assert torch.equal(g[name][k], v[0]), (k, name, g[name][k], v[0])
