"""Device memory that is used again: blocks of nh_device_alloc and the arrays
of a rebuilt Hamiltonian."""
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


def test_freed_blocks_are_reused_and_bounded():
    H = Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=None)
    size = 3 << 20
    a = native.DeviceArray(H, size, dtype=np.uint8)
    b = native.DeviceArray(H, size, dtype=np.uint8)
    pa, pb, idle = a.ptr.value, b.ptr.value, mem_info(H)[1]
    assert pa != pb
    a.free()
    assert mem_info(H)[1] == idle + size
    c = native.DeviceArray(H, size + 1, dtype=np.uint8)  # another size: another block
    assert c.ptr.value not in (pa, pb)
    d = native.DeviceArray(H, size, dtype=np.uint8)
    assert d.ptr.value == pa and mem_info(H)[1] == idle
    d.upload(np.arange(size, dtype=np.uint8))
    assert np.array_equal(d.download(), np.arange(size, dtype=np.uint8))
    many = [native.DeviceArray(H, size, dtype=np.uint8) for _ in range(12)]
    for m in many:
        m.free()
    assert mem_info(H)[1] == idle + 8 * size
    # a block above the bound goes back to the device at once
    fr = mem_info(H)[0]
    big = native.DeviceArray(H, fr // 16, dtype=np.uint8)
    big.free()
    assert mem_info(H)[1] == idle + 8 * size
    b.free()
    c.free()
    H.close()


def test_rebuild_in_other_layouts_equals_a_fresh_build():
    M = _models.gaas_box(cells=(2, 3, 1), strain_nm=0.02, seed=4, alloy=True)
    H = Hamiltonian(M, layout=native.LAYOUT_SK)
    x = _models.random_vectors(H.n, 1, seed=5)[0]
    for layout, prec in ((native.LAYOUT_SK, native.PREC_FP32),
                         (native.LAYOUT_BLOCKS, native.PREC_FP64),
                         (native.LAYOUT_BLOCKS, native.PREC_FP32),
                         (native.LAYOUT_MATRIX_FREE, native.PREC_FP64),
                         (native.LAYOUT_SK, native.PREC_FP64),
                         (native.LAYOUT_SK, native.PREC_FP64)):
        print(layout, prec, flush=True)
        H.build(layout, prec)
        F = Hamiltonian(M, layout=layout, precision=prec)
        assert np.array_equal(H.hv(x, 0.3), F.hv(x, 0.3))
        F.close()
    with pytest.raises(native.NHError):
        native.check(native.load().nh_ham_export(H.ctx, native.ptr(np.zeros(17 * M.n_atoms)),
                                                 None))
