"""The autotuner's trials form their sums the way the whole call does."""
from ctypes import byref, c_int, c_void_p

import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth


def _args(dtype, pgram, nf=1000000, K=200, n=30000):
    a = _native.SweepArgs()
    a.variant, a.dtype, a.form = _native.STANDARD, dtype, _native.FORM_SPLIT32
    a.num_objects, a.num_freqs, a.num_obs, a.top_k = K, nf, n, 1
    a.min_freq, a.max_freq = synth.OMEGA_MIN, synth.OMEGA_MAX
    a.pgram = 4096 if pgram else None  # never dereferenced
    return a


def test_trials_of_coarse_sums_have_a_periodogram():
    """FP32 periodograms on a fine grid: the trials write one of 65536 bins,
    into the workspace.  Direct sums (FP64, or few terms) and peaks alone need none."""
    L = _native.core()
    size = lambda *a, **k: L.lsamd_autotune_workspace_size(byref(_args(*a, **k)))
    assert size(_native.F32, True) - size(_native.F32, False) >= 4 * 200 * 65536
    assert size(_native.F64, True) == size(_native.F64, False)
    assert size(_native.F32, True, nf=40000) == size(_native.F32, False, nf=40000)


@pytest.mark.gpu
@pytest.mark.parametrize("pgram", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nf", [20001, 500009])
def test_autotune_leaves_outputs_alone(nf, dtype, pgram):
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    b = synth.lognormal_batch(200, 140, 0.6, 20, 1000, 1800, False, 46)
    plan = device.SweepPlan(*device.numpy_to_device(b["obj_id"], b["t"], b["y"], None, dtype), min_freq=synth.OMEGA_MIN,
                            max_freq=synth.OMEGA_MAX, num_freqs=nf, variant=_native.STANDARD,
                            form=_native.FORM_SPLIT32, top_k=3, pgram=pgram)
    plan.run()
    ref = {k: v.clone() for k, v in plan.results().items()}
    # a workspace without room for a trial's periodogram is taken as well
    T, M = c_int(), c_int()
    assert plan.lib.lsamd_autotune(byref(plan.args), c_void_p(plan.workspace.data_ptr()), plan.workspace.numel(),
                                   c_void_p(torch.cuda.current_stream().cuda_stream), byref(T), byref(M)) == _native.OK
    assert plan.autotune() == plan.tile()
    for k, v in plan.results().items():
        assert torch.equal(v, ref[k]), k
