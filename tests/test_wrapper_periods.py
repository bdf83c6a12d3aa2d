"""Periods of the Python wrapper for every kind of number that a grid is given in (CPU)."""
import numpy as np
import pytest

from gpu_lomb_scargle_amd import lombscarglegpu as ls


@pytest.mark.parametrize("kind", [float, np.float64, np.float32, np.float16])
@pytest.mark.parametrize("nf", [4003, np.int64(4003)])
def test_periods_are_formed_from_numpy_s_argmax(kind, nf):
    """A NumPy scalar keeps its precision when multiplied by a Python int, and
    widens with argmax's int64: FP32 frequencies give FP64 periods."""
    rng = np.random.default_rng(3)
    o = np.repeat([4, 9], 60)
    t = np.concatenate([np.sort(rng.uniform(0, 200, 60)) for _ in range(2)])
    y = np.sin(2.0 * t) + rng.normal(0, 0.3, 120)
    lo, hi = kind(0.1), kind(3.0)
    _, periods, pgram = ls.lombscargle(o, t, y, lo, hi, False, "CPU", None, nf, "double")
    df = (hi - lo) / nf * 1.0
    want = [1.0 / (lo + (df * np.argmax(row))) for row in pgram]
    assert np.array_equal(periods, want)
