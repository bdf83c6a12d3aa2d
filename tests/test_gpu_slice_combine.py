"""The combiner of a single object's observation slices, over tiles whose bins
per thread it spreads over 2 to 16 groups of threads (M = 3 to 16, one and
several wavefronts per group), ragged chunks and few or many slices: against
the same object swept without slices.

Tolerances: the sums are regrouped only.  split: FP64 sums, 1e-12.  split32:
each side within 1e-5 of the FP64 power on bins of at least 1e-3 Pmax (2e-6
Pmax on all), so 2e-5 and 4e-6 between them.  The peaks are the first maxima
of the sliced periodogram itself, exactly."""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth
from test_gpu_parity import F64, _one_object, assert_close

pytestmark = pytest.mark.gpu
S, G = _native.STANDARD, _native.GENERALIZED


@pytest.mark.parametrize("n", [130, 3555])
@pytest.mark.parametrize("form,variant,tile", [
    (_native.FORM_SPLIT, S, (256, 16)), (_native.FORM_SPLIT, S, (256, 14)), (_native.FORM_SPLIT, S, (512, 8)),
    (_native.FORM_SPLIT, S, (128, 8)), (_native.FORM_SPLIT, G, (256, 2)), (_native.FORM_SPLIT32, S, (64, 16)),
    (_native.FORM_SPLIT32, S, (64, 6)), (_native.FORM_SPLIT32, G, (64, 16)), (_native.FORM_SPLIT32, G, (256, 3))])
def test_sliced_against_whole(form, variant, tile, n):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    t, y, dy = _one_object(variant)
    t, y, dy = t[:n], y[:n], None if dy is None else dy[:n]
    nf = 20011
    d = device.numpy_to_device(np.zeros(n, np.uint32), t, y, dy, F64)
    out = []
    for slices in (0, 1):
        p = device.SweepPlan(*d, min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MAX, num_freqs=nf, variant=variant,
                             form=form, top_k=3, tile=tile, obs_slices=slices)
        p.run()
        torch.cuda.synchronize()
        out.append({k: v.cpu().numpy() for k, v in p.results().items()})
    a, b = (o["pgram"][0] for o in out)
    if form == _native.FORM_SPLIT:
        assert_close(a, b, 1e-12, 1e-3, 1e-12)
    else:
        assert_close(a, b, 2e-5, 1e-3, 4e-6)
    best = np.lexsort((np.arange(nf), -a))[:3]
    assert np.array_equal(out[0]["index"][0], best) and np.array_equal(out[0]["power"][0], a[best])
