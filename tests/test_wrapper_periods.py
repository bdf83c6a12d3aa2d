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


def test_a_peak_at_frequency_zero_has_an_infinite_period():
    """0/0 at frequency 0 is numpy's argmax; the period is inf, with numpy's
    warning, as the loop over numpy scalars had it."""
    rng = np.random.default_rng(4)
    t = np.sort(rng.uniform(0, 200, 60))
    with pytest.warns(RuntimeWarning, match="divide by zero"):
        _, periods, pgram = ls.lombscargle(np.zeros(60, int), t, np.sin(2.0 * t), 0.0, 3.0, False, "CPU", None, 2003, "double")
    assert np.isnan(pgram[0, 0]) and np.isinf(periods[0])
