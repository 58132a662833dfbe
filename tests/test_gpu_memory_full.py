"""Allocations of the library on a device that is full but for idle blocks of its
own: they are handed back, whatever allocation asks."""
import numpy as np
import pytest
import torch

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import refine_eigenpairs

pytestmark = pytest.mark.gpu


def fill_device(leave):
    """Everything but less than `leave` bytes, in torch's hands."""
    held = []
    size = max(torch.cuda.mem_get_info()[0] - leave, leave)
    while size >= leave:
        try:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.cuda.OutOfMemoryError:
            size //= 2
    return held


@pytest.mark.parametrize("layout", [native.LAYOUT_SK, native.LAYOUT_MATRIX_FREE])
def test_first_build_takes_back_idle_workspace(layout):
    """The first SK or matrix-free build makes the block tables (36 MB here)
    beside the Hamiltonian; with next to nothing free (8 MB and what torch cannot
    take in one piece) and 1 GB idle in another context it succeeds."""
    small = _models.gaas_box(cells=(15, 15, 14), seed=3)
    idle = Hamiltonian(small, layout=native.LAYOUT_SK)
    H = Hamiltonian(_models.gaas_box(cells=(46, 46, 46)), layout=None)
    refine_eigenpairs(idle, _models.random_vectors(idle.n, 8, seed=4), np.linspace(0.5, 1.5, 8),
                      depth=12, max_rounds=1)
    held = fill_device(8 << 20)
    print("free %.1f MB" % (torch.cuda.mem_get_info()[0] / 1e6), flush=True)
    try:
        H.build(layout)
    finally:
        del held
        torch.cuda.empty_cache()
    x = native.DeviceArray.from_host(H, np.ones(H.n, dtype=np.complex128))
    y = H.hv(x).download()
    assert np.isfinite(y).all() and np.abs(y).max() > 1.0
    H.close()
    idle.close()
