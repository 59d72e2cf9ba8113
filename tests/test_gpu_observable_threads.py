"""Observables of one field read through the C ABI from several threads: each thread gets its own,
as read alone.  (Python's getters hold the interpreter's lock; calls through ctypes overlap.)"""
import ctypes
import os
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Options(ctypes.Structure):
    _fields_ = [("precision", ctypes.c_int), ("seed", ctypes.c_uint64), ("timestep", ctypes.c_int64),
                ("tile", ctypes.c_int)]


# one staging piece a component, and several and a part
@pytest.mark.parametrize("shape", [(256, 512), (1000, 513)])
def test_observables_from_threads(shape):
    lib = ctypes.CDLL(os.path.join(REPO, "active-model-bplus_amd", "lib", "libamb.so"))

    def ptr(a):
        return ctypes.c_void_p(a.ctypes.data)

    def get(which):
        out = np.zeros((2,) + shape)
        if which < 0:
            assert lib.amb_get_field(h, ptr(out)) == 0
        else:
            assert lib.amb_get_observable(h, which, ptr(out)) == 0
        return out

    phi = 0.05 * np.random.default_rng(4).normal(size=shape)
    stencil, model = (ctypes.c_double * 3)(5e-3, 1, 1), (ctypes.c_double * 7)(-0.25, 0, 0.25, 1, 0.5, -1, 0.05)
    opt, h = Options(64, 1, 0, 0), ctypes.c_void_p()
    assert lib.amb_create(ptr(phi), ctypes.c_int64(shape[0]), ctypes.c_int64(shape[1]), stencil, model,
                          ctypes.byref(opt), ctypes.byref(h)) == 0
    try:
        which = [-1, 0, 3, 2, 9, 8]  # the field, two potentials, three currents
        together = [None] * len(which)

        def read(i):
            together[i] = get(which[i])

        threads = [threading.Thread(target=read, args=(i,)) for i in range(len(which))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for i, w in enumerate(which):
            np.testing.assert_array_equal(together[i], get(w), err_msg=str(w))
    finally:
        lib.amb_destroy(h)
