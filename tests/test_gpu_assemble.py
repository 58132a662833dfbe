"""Assembly of every layout against the oracle's dense matrix: atom counts
that are no multiple of a workgroup's 32, absent neighbours with and without
passivation, alloys, large strain (the corrections then reach tenths of an
eV), a potential, 10 and 20 bands."""
import numpy as np
import pytest

import _models
from nemo3d_amd import materials, native
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import oracle

pytestmark = pytest.mark.gpu

LAYOUTS = {"blocks": native.LAYOUT_BLOCKS, "sk": native.LAYOUT_SK,
           "mf": native.LAYOUT_MATRIX_FREE}
CASES = {
    "strained": dict(cells=(2, 1, 1), strain_nm=0.04, seed=21),
    "alloy_phi": dict(cells=(1, 1, 2), strain_nm=0.02, seed=22, alloy=True, phi=True),
    "open": dict(cells=(1, 2, 1), strain_nm=0.03, seed=23, passivate=False),
    "ten_bands": dict(cells=(2, 2, 1), strain_nm=0.03, seed=24, alloy=True,
                      band=materials.BANDS_10_NOSPIN),
}


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("case", sorted(CASES))
def test_dense_matrix(case, layout):
    """Entries to 1e-12 of the largest (the bound of the other assembly
    tests), exactly Hermitian, and the same after a rebuild."""
    M = _models.gaas_box(**CASES[case])
    ref = oracle.assemble(M.arrays()).dense()
    H = Hamiltonian(M, layout=LAYOUTS[layout])
    print(case, layout, "N", H.n, flush=True)
    dX = native.DeviceArray.from_host(H, np.eye(H.n, dtype=np.complex128))
    D = H.hV(dX, 0.0).download().T
    assert np.abs(D - ref).max() <= 1e-12 * np.abs(ref).max()
    if layout != "blocks":
        assert np.array_equal(D, D.conj().T)
    H.build(LAYOUTS[layout])
    assert np.array_equal(H.hV(dX, 0.0).download().T, D)
