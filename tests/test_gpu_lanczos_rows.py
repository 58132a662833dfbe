"""Lanczos steps on stored blocks about the sizes where a workgroup takes more
wavefronts, against the same recurrence with the device's products (FP64: the
step's FP32 products round the vector before it is normalised)."""
import numpy as np
import pytest

import _models
from nemo3d_amd import materials, native
from nemo3d_amd.hamiltonian import Hamiltonian
from test_gpu_sk_blocks import device_tridiagonal, tridiagonal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [materials.BANDS_20_SPIN, materials.BANDS_10_NOSPIN])
@pytest.mark.parametrize("cells", [(12, 8, 8), (1, 769, 1), (12, 12, 8), (1, 1153, 1),
                                   (16, 12, 8), (29, 53, 1)])
def test_steps_match_recurrence(cells, band):
    """6,144 and 6,152, 9,216 and 9,224, 12,288 and 12,296 atoms; bound as for the
    one-launch step (rounding of |H| < 40 eV, amplified by |H| / beta < 10 in
    each of 8 steps)."""
    H = Hamiltonian(_models.gaas_box(cells=cells, strain_nm=0.005, seed=8, band=band),
                    layout=native.LAYOUT_BLOCKS)
    print(H.n_atoms, flush=True)
    q = _models.random_vectors(H.n, 1, seed=9)[0]
    q /= np.linalg.norm(q)
    a, b = device_tridiagonal(H, q, 8)
    ar, br = tridiagonal(H, q, 8)
    assert np.abs(a - ar).max() < 1e-9 and np.abs(b - br).max() < 1e-9
