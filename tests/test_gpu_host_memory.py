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
