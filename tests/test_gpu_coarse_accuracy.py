"""FP32 periodograms on the coarse grid are no further from FP64 than the direct
sums: few observations and every oversampling between one coarse step and the
next, where the window's aliasing would show.

Both against the plain FP64 form on the same float inputs, over the bins of at
least 1e-3 of the peak of 24 objects.  The root of the mean squared relative
error may be 1.2 times the direct sums': equal but for the scatter of the few
bins that carry it (the window used at its own least oversampling has 1.5 to
3.4)."""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth

pytestmark = pytest.mark.gpu
F32, F64 = np.float32, np.float64
DF = (synth.OMEGA_MAX - synth.OMEGA_MIN) / (2 * np.pi)  # cycles/day of the whole grid
K, NF = 24, 262147


def _curves(n, over, gen, seed):
    rng = np.random.default_rng(seed)
    span = NF / DF / over
    ts, ys, ds = [], [], []
    for _ in range(K):
        t = np.sort(np.floor(rng.uniform(0, span, n)) + rng.uniform(0, 0.3, n))
        t[0], t[-1] = 0.0, span
        y = 0.5 * np.sin(2 * np.pi * rng.uniform(0.3, 20.0) * t) + rng.normal(0, 0.3, n)
        ts.append(t.astype(F32))
        ys.append((y + (17 if gen else 0)).astype(F32))
        ds.append(np.exp(rng.uniform(np.log(0.01), np.log(0.2), n)).astype(F32))
    o = np.repeat(np.arange(K, dtype=np.uint32), n)
    return o, np.concatenate(ts), np.concatenate(ys), np.concatenate(ds) if gen else None


def _sweep(o, t, y, dy, dtype, form, gen, **kw):
    from gpu_lomb_scargle_amd import device
    return device.sweep(*device.numpy_to_device(o, t, y, dy, dtype), min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MAX,
                        num_freqs=NF, form=form, variant=_native.GENERALIZED if gen else _native.STANDARD, top_k=1,
                        **kw)["pgram"].double()


@pytest.mark.parametrize("gen", [False, True], ids=["standard", "generalized"])
@pytest.mark.parametrize("n", [34, 60, 120])
@pytest.mark.parametrize("h", [4, 8])
@pytest.mark.parametrize("sigma", [1.96, 2.1, 2.33, 2.41, 2.6])
def test_error_against_the_direct_sums(sigma, h, n, gen):
    torch = pytest.importorskip("torch")
    c = _curves(n, sigma * h, gen, 100 * n + h)
    ref = _sweep(*c, F64, _native.FORM_PLAIN, gen)
    coarse = _sweep(*c, F32, _native.FORM_SPLIT32, gen, obs_slices=1)
    direct = _sweep(*c, F32, _native.FORM_SPLIT32, gen)  # under 1.5e9 terms
    big = ref >= 1e-3 * ref.max(1, keepdim=True).values
    e = [torch.sqrt((((p - ref) / ref)[big] ** 2).mean()).item() for p in (coarse, direct)]
    print(f"coarse {e[0]:.2e} direct {e[1]:.2e}")
    assert e[0] <= 1.2 * e[1]


@pytest.mark.parametrize("n,coarse", [(8192, True), (8193, False)])
def test_generalized_objects_of_many_observations_keep_the_direct_sums(n, coarse):
    """Their y sums are folded in FP64 there.  Five objects are under the terms of
    the coarse grid, 24 are above."""
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    o, t, y, dy = _curves(n, 2.5 * 4, True, n)
    kw = dict(min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MIN + (synth.OMEGA_MAX - synth.OMEGA_MIN) * 20001 / NF,
              num_freqs=20001, form=_native.FORM_SPLIT32, variant=_native.GENERALIZED, top_k=1)
    whole = device.sweep(*device.numpy_to_device(o, t, y, dy, F32), **kw)["pgram"]
    few = device.sweep(*device.numpy_to_device(o[:5 * n], t[:5 * n], y[:5 * n], dy[:5 * n], F32), **kw)["pgram"]
    assert torch.equal(whole[:5], few) == (not coarse)
