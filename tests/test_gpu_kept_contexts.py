"""Freed device arrays that contexts keep, over several contexts."""
import ctypes

import numpy as np
import pytest

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian

pytestmark = pytest.mark.gpu


def mem_info(H):
    fr, idle = ctypes.c_int64(), ctypes.c_int64()
    native.check(native.load().nh_context_mem_info(H.ctx, ctypes.byref(fr), ctypes.byref(idle)))
    return fr.value, idle.value


def test_bound_holds_over_contexts():
    """Three contexts that each free a 50th of the memory keep no more than a
    32nd of it, and nothing when they are gone."""
    Hs = [Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=None) for _ in range(3)]
    fr, idle = mem_info(Hs[0])
    arrays = [native.DeviceArray(H, fr // 50, dtype=np.uint8) for H in Hs]
    for a in arrays:
        a.free()
    kept = mem_info(Hs[0])[1] - idle
    print("kept %.2f of a 32nd" % (kept / (fr / 32)), flush=True)
    assert fr // 50 <= kept <= 1.05 * fr / 32
    for H in Hs[1:]:
        H.close()
    last = Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=None)
    assert mem_info(last)[1] <= kept
    Hs[0].close()
    last.close()


def test_second_free_through_another_context_is_refused():
    A = Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=None)
    B = Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=None)
    lib = native.load()
    p = ctypes.c_void_p()
    native.check(lib.nh_device_alloc(A.ctx, 4096, ctypes.byref(p)))
    native.check(lib.nh_device_free(A.ctx, p))
    with pytest.raises(native.NHError):
        native.check(lib.nh_device_free(B.ctx, p))
    B.close()
    q = ctypes.c_void_p()  # the block is A's still
    native.check(lib.nh_device_alloc(A.ctx, 4096, ctypes.byref(q)))
    assert q.value == p.value
    native.check(lib.nh_device_free(A.ctx, q))
    A.close()
