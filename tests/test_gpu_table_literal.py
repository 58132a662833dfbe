"""The Slater-Koster table's literal sqrt 3 (1e-12 off) in every layout: products
of strained alloys agree with the oracle, and the layouts with each other, to
rounding; so do the onsite records."""
import numpy as np
import pytest

import _models
from nemo3d_amd import materials, native
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import oracle

pytestmark = pytest.mark.gpu

LAYOUTS = [native.LAYOUT_BLOCKS, native.LAYOUT_SK, native.LAYOUT_MATRIX_FREE]


@pytest.mark.parametrize("band", [materials.BANDS_20_SPIN, materials.BANDS_10_NOSPIN])
@pytest.mark.parametrize("strain", [0.0, 0.004, 0.02])
def test_products_to_rounding(band, strain):
    """Relative 2-norm: a bond's product is rounded about 20 times (each 1.1e-16,
    of random sign), its integrals and the oracle's a few times each: 5e-16 to
    1e-15; three times that."""
    M = _models.gaas_box(cells=(3, 2, 2), strain_nm=strain, seed=11, alloy=True, band=band)
    ref = oracle.assemble(M.arrays())
    X = _models.random_vectors(ref.n, 2, seed=12)
    Yr = np.array([ref.hv(x, 0.3) for x in X])
    Y = {}
    for layout in LAYOUTS:
        H = Hamiltonian(M, layout=layout)
        Y[layout] = np.array(H.hV(X, 0.3))
        err = np.linalg.norm(Y[layout] - Yr) / np.linalg.norm(Yr)
        print(layout, "strain", strain, "error %.2e" % err, flush=True)
        assert err < 3e-15
    for layout in LAYOUTS[1:]:
        d = np.linalg.norm(Y[layout] - Y[LAYOUTS[0]]) / np.linalg.norm(Yr)
        assert d < 3e-15


def test_onsite_records_to_rounding():
    """Absolute, eV: sums of about 40 terms below 20 eV, each rounded to 1e-16 of
    it and of random sign: 2e-14."""
    M = _models.gaas_box(cells=(3, 2, 2), strain_nm=0.02, seed=13, alloy=True)
    ref = oracle.assemble(M.arrays())
    onsite = Hamiltonian(M, layout=native.LAYOUT_BLOCKS).export()[0]
    d = np.abs(onsite - np.asarray(ref.onsite)[:, :17])
    print("onsite: largest difference %.2e eV" % d.max(), flush=True)
    assert d.max() < 2e-14
