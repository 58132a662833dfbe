"""The Slater-Koster table's literal sqrt 3 (1e-12 off): the onsite records of a
strained alloy agree with the oracle's to rounding."""
import numpy as np
import pytest

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import oracle

pytestmark = pytest.mark.gpu

def test_onsite_records_to_rounding():
    """Absolute, eV: sums of about 40 terms below 20 eV, each rounded to 1e-16 of
    it and of random sign: 2e-14."""
    M = _models.gaas_box(cells=(3, 2, 2), strain_nm=0.02, seed=13, alloy=True)
    ref = oracle.assemble(M.arrays())
    onsite = Hamiltonian(M, layout=native.LAYOUT_BLOCKS).export()[0]
    d = np.abs(onsite - np.asarray(ref.onsite)[:, :17])
    print("onsite: largest difference %.2e eV" % d.max(), flush=True)
    assert d.max() < 2e-14
