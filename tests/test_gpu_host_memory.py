"""What host calls leave of the caller's memory and in their own."""
import ctypes
import mmap

import numpy as np
import pytest

from gpu_lomb_scargle_amd import _native, synth

pytestmark = pytest.mark.gpu


def _vm_flags(address):
    """VmFlags of the mapping that holds the address."""
    inside = False
    for line in open("/proc/self/smaps"):
        head = line.split()[0]
        if "-" in head and not head.endswith(":"):
            a, b = (int(x, 16) for x in head.split("-"))
            inside = a <= address < b
        elif inside and line.startswith("VmFlags"):
            return line.split()[1:]
    return []


def test_the_page_policy_of_the_output_stays_the_callers():
    b = synth.lognormal_batch(40, 50, 0.3, 5, 200, 1800, False, 31)
    nf = 100003
    room = mmap.mmap(-1, 40 * nf * 8)
    at = ctypes.addressof(ctypes.c_char.from_buffer(room))
    middle = at + 20 * nf * 8
    before = _vm_flags(middle)
    L = _native.core()
    o = np.ascontiguousarray(b["obj_id"], np.uint32)
    t, y = (np.ascontiguousarray(b[k], np.float64) for k in "ty")
    rc = L.lsamd_batch_host(_native.STANDARD, _native.F64, _native.FORM_SPLIT32, 1, 1, _native.ptr(o), _native.ptr(t),
                            _native.ptr(y), None, len(t), synth.OMEGA_MIN, synth.OMEGA_MAX, nf, ctypes.c_void_p(at), 0, None,
                            None, None, None)
    _native.check(L, rc)
    pgram = np.frombuffer(room, np.float64)
    assert pgram.max() > 0
    assert before and _vm_flags(middle) == before


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_calls_of_all_sizes_in_turn(dtype, monkeypatch):
    """Periodograms of 288 MB and more (staged copies of device memory), of 32 MB
    and 160 MB (slices swept into pinned memory), of 40 kB (one piece), then all
    again, whole and in smaller slices: each equals the sweep of device tensors."""
    torch = pytest.importorskip("torch")
    from gpu_lomb_scargle_amd import device
    b = synth.lognormal_batch(40, 30, 0.3, 5, 100, 1800, False, 31)
    o, t, y = b["obj_id"], b["t"], b["y"]
    wide = 8 // np.dtype(dtype).itemsize
    ref = {}
    for nf in (900007 * wide, 100003, 1250 * wide, 500009 * wide):
        p = device.SweepPlan(*device.numpy_to_device(o, t, y, None, dtype), min_freq=synth.OMEGA_MIN, max_freq=synth.OMEGA_MAX,
                             num_freqs=nf, variant=_native.STANDARD, form=_native.FORM_SPLIT32, top_k=3, obs_slices=1)
        p.run()
        torch.cuda.synchronize()
        ref[nf] = {k: v.cpu().numpy() for k, v in p.results().items()}
        del p
    for slices in (None, 20 << 20, 3 << 20):
        if slices:
            monkeypatch.setenv("LSAMD_SLICE_BYTES", str(slices))
        for nf, want in ref.items():
            r = _native.batch_host(o, t, y, None, synth.OMEGA_MIN, synth.OMEGA_MAX, nf, _native.STANDARD, dtype,
                                   _native.FORM_SPLIT32, top_k=3)
            for k in ("pgram", "index", "power", "period"):
                assert np.array_equal(np.asarray(r[k]), want[k].astype(np.asarray(r[k]).dtype)), (nf, slices, k)
