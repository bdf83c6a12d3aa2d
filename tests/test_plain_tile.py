"""The plain standard FP64 sweep's tile: chosen by the grid, or the caller's (CPU
for the workspace sizes, GPU for the bits)."""
from ctypes import byref, c_int

import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth

F64 = np.float64


def _args(K, nf, n, tile=(0, 0), obs_slices=0):
    a = _native.SweepArgs()
    a.variant, a.dtype, a.form = _native.STANDARD, _native.F64, _native.FORM_PLAIN
    a.num_objects, a.num_freqs, a.num_obs, a.top_k = K, nf, n, 3
    a.min_freq, a.max_freq = 1.0, 100.0
    a.tile_threads, a.tile_fpt = tile
    a.obs_slices = obs_slices
    return a


def test_a_workspace_serves_smaller_calls():
    """The workspace of a call is enough for every call of fewer objects, bins or
    observations, whatever kernel those take."""
    L = _native.core()
    grids = [1, 255, 256, 257, 4096, 8191, 8192, 8193, 40000, 147455, 147456, 262144, 1000003]
    counts = [1, 2, 3, 9, 10, 11, 200]
    for obs_slices in (0, 1):
        size = {(K, nf): L.lsamd_sweep_workspace_size(byref(_args(K, nf, 5000, obs_slices=obs_slices)))
                for K in counts for nf in grids}
        for (K, nf), s in size.items():
            for (k, f), less in size.items():
                assert k > K or f > nf or less <= s, (K, nf, k, f, obs_slices)


def _tile(a):
    T, M = c_int(), c_int()
    _native.core().lsamd_sweep_tile(byref(a), byref(T), byref(M))
    return T.value, M.value


def test_the_tile_that_runs():
    """A tile that the caller names, for the call or for the process, is the one
    that runs; the built-in one follows the bins per object, and only the split
    of the same chains over threads the number of objects."""
    L = _native.core()
    for K in (2, 100, 100000):
        assert _tile(_args(K, 8191, 50 * K)) == (256, 1)
        assert _tile(_args(K, 8192, 50 * K)) == ((256, 8) if K < 256 else (256, 16))
    assert _tile(_args(1, 147455, 50)) == (256, 1) and _tile(_args(1, 147456, 50)) == (256, 8)
    assert _tile(_args(1, 8192, 50, obs_slices=1)) == (256, 8)
    for tile in ((256, 1), (256, 2), (256, 8), (256, 16)):
        assert _tile(_args(3, 1000000, 150, tile)) == tile
    a = _args(3, 1000000, 150)
    assert _tile(a) == (256, 16)
    try:
        assert L.lsamd_set_tile(a.form, a.variant, 256, 1) == _native.OK
        assert _tile(a) == (256, 1)
    finally:
        L.lsamd_set_tile(a.form, a.variant, 0, 0)
    assert L.lsamd_set_tile(a.form, a.variant, 256, 16) == _native.ERR_INVALID  # no FP32 kernel of that shape
    a.dtype = _native.F32
    assert _tile(a) == (256, 1)


def _curves(counts, seed=3):
    rng = np.random.default_rng(seed)
    ts = [np.sort(rng.integers(0, 1800, n) + rng.uniform(0, 0.3, n)) for n in counts]
    ys = [np.sin(3.1 * t) + rng.normal(0, 0.3, len(t)) for t in ts]
    return np.repeat(np.arange(len(counts), dtype=np.uint32), counts), np.concatenate(ts), np.concatenate(ys)


def _sweep(o, t, y, lo, hi, nf, **kw):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    p = device.SweepPlan(*device.numpy_to_device(o, t, y, None, F64), min_freq=lo, max_freq=hi, num_freqs=nf,
                         variant=_native.STANDARD, form=_native.FORM_PLAIN, top_k=3, **kw)
    p.run()
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in p.results().items()}, p.tile()


@pytest.mark.gpu
@pytest.mark.parametrize("schedule", [_native.SCHEDULE_GRID, _native.SCHEDULE_PERSISTENT])
@pytest.mark.parametrize("lo,hi", [(synth.OMEGA_MIN, synth.OMEGA_MAX), (-20.0, 40.0), (1e-4, 60.0)])
@pytest.mark.parametrize("nf", [8192, 8193, 20479, 20480, 20481, 40013])
def test_whole_and_half_chains_have_the_same_bits(nf, lo, hi, schedule):
    """Ragged chunks, grids over and near zero, few observations, one
    observation past the steps' range, a NaN and equal times, equal powers."""
    o, t, y = _curves([5, 15, 16, 17, 255, 256, 257, 300, 300, 300, 60])
    t[o == 7] = np.where(np.arange(300) == 250, 2.0 ** 28 / 1.1, t[o == 7])
    t[o == 8] = 3.5
    t[np.nonzero(o == 9)[0][3]] = np.nan
    y[o == 10] = 0.0
    (a, ta), (b, tb) = (_sweep(o, t, y, lo, hi, nf, schedule=schedule, tile=tile) for tile in ((256, 8), (256, 16)))
    assert (ta, tb) == ((256, 8), (256, 16))
    for key in a:
        assert np.array_equal(a[key], b[key], equal_nan=True), key


@pytest.mark.gpu
@pytest.mark.parametrize("nf", [5003, 8192, 30011])
def test_an_objects_powers_do_not_depend_on_the_others(nf):
    """The first stars of a call of 300, alone in a call of 2 and of 20, on the
    device and through the host call; alone with obs_slices = 1."""
    o, t, y = _curves([90] * 300)
    whole, _ = _sweep(o, t, y, 1.0, 60.0, nf)
    host = _native.batch_host(o, t, y, None, 1.0, 60.0, nf, _native.STANDARD, F64, _native.FORM_PLAIN)["pgram"]
    assert np.array_equal(host, whole["pgram"])
    for K in (2, 20):
        part, _ = _sweep(o[:90 * K], t[:90 * K], y[:90 * K], 1.0, 60.0, nf)
        for key in part:
            assert np.array_equal(part[key], whole[key][:K]), (key, K)
        host = _native.batch_host(o[:90 * K], t[:90 * K], y[:90 * K], None, 1.0, 60.0, nf, _native.STANDARD, F64,
                                  _native.FORM_PLAIN)["pgram"]
        assert np.array_equal(host, whole["pgram"][:K])
    one, _ = _sweep(o[:90], t[:90], y[:90], 1.0, 60.0, nf, obs_slices=1)
    assert np.array_equal(one["pgram"][0], whole["pgram"][0])


@pytest.mark.gpu
def test_a_named_tile_runs_its_kernel():
    """256 x 1 asked for by name: a sine and cosine per bin, as 256 x 2 has them."""
    o, t, y = _curves([90] * 20)
    a, b = (_sweep(o, t, y, 1.0, 60.0, 40013, tile=tile)[0] for tile in ((256, 1), (256, 2)))
    assert np.array_equal(a["pgram"], b["pgram"])


@pytest.mark.gpu
@pytest.mark.parametrize("K,nf,tile", [(1, 100003, "256x1"), (1, 200003, "256x8"), (3, 5003, "256x1"), (3, 20011, "256x8")])
def test_the_stats_record_names_the_tile(K, nf, tile, tmp_path, monkeypatch):
    from gpu_lomb_scargle_amd import lombscarglegpu as ls
    monkeypatch.chdir(tmp_path)
    monkeypatch.setenv("LSAMD_GPU_STATS", "1")
    o, t, y = _curves([40] * K)
    ls.lombscargle(o, t, y, 0.1, 10.0, False, "GPU", None, nf, "double")
    assert (tmp_path / "gpu_stats.txt").read_text().strip().endswith(tile)
