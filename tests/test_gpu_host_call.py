"""Host calls around the sizes where the way of their inputs and outputs
changes: outputs the kernels write into pinned memory (up to 256 KiB), one copy
of the whole (up to 8 MiB), slices with staged copies; inputs packed (up to
1 MiB) or copied one by one; peaks alone, and calls that follow a larger or
smaller one.  The same observations through device tensors give the same bits,
and the row maxima equal numpy's."""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth
from gpu_lomb_scargle_amd import lombscarglegpu as ls

pytestmark = pytest.mark.gpu
F32, F64 = np.float32, np.float64


def _curves(K, n, gen):
    b = synth.lognormal_batch(K, n, 0.3, 5, 4 * n, 1800, gen, 31)
    return b["obj_id"], b["t"], b["y"], b["dy"] if gen else None


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("K,n,nf", [(1, 29, 1188), (7, 40, 9361), (8, 40, 8192), (3, 50, 300007), (40, 60, 30011),
                                    (300, 400, 4001), (2, 9, 5)])
def test_against_device_tensors(K, n, nf, dtype):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    o, t, y, _ = _curves(K, n, False)
    args = (o, t, y, None, synth.OMEGA_MIN, synth.OMEGA_MAX, nf, _native.STANDARD, dtype, _native.FORM_SPLIT)
    r = _native.batch_host(*args, top_k=3)
    p = device.SweepPlan(*device.numpy_to_device(o, t, y, None, dtype), min_freq=synth.OMEGA_MIN, top_k=3,
                         max_freq=synth.OMEGA_MAX, num_freqs=nf, variant=_native.STANDARD, form=_native.FORM_SPLIT,
                         obs_slices=0 if K == 1 else 1)
    p.run()
    torch.cuda.synchronize()
    d = {k: v.cpu().numpy() for k, v in p.results().items()}
    for key in ("pgram", "index", "power", "period"):
        assert np.array_equal(np.asarray(r[key]), d[key].astype(np.asarray(r[key]).dtype)), key
    alone = _native.batch_host(*args, top_k=3, pgram=False)
    for key in ("index", "power", "period"):
        assert np.array_equal(alone[key], r[key]), key


@pytest.mark.parametrize("dtype", ["float", "double"])
def test_wrapper_periods(dtype):
    """A call of 12 stars, a larger one, and the first again: the same bits, and
    periods from numpy's argmax of the rows."""
    small, large = _curves(12, 50, True), _curves(60, 50, True)
    runs = []
    for (o, t, y, dy), nf in ((small, 20001), (large, 60001), (small, 20001)):
        ids, periods, pg = ls.lombscargle(o, t, y.copy(), 0.1, 10.0, True, "GPU", dy, nf, dtype)
        df = (10.0 - 0.1) / nf * 1.0
        assert np.array_equal(periods, [1.0 / (0.1 + df * int(np.argmax(row))) for row in pg])
        runs.append((ids, periods, pg))
    for a, b in zip(runs[0], runs[2]):
        assert np.array_equal(a, b)
