"""Stored-block products, six atoms a wavefront and 24 a workgroup: atom counts
around those, absent neighbours, both precisions and band counts, against the
oracle; and the Lanczos step built on them against the written-out recurrence."""
import numpy as np
import pytest

import _models
from nemo3d_amd import materials, native
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import oracle
from test_gpu_sk_blocks import device_tridiagonal, tridiagonal

pytestmark = pytest.mark.gpu

BANDS = {20: materials.BANDS_20_SPIN, 10: materials.BANDS_10_NOSPIN}


@pytest.mark.parametrize("bands", [10, 20])
@pytest.mark.parametrize("cells,passivate", [((1, 1, 1), True), ((3, 1, 1), False),
                                             ((5, 5, 1), True)])
def test_rows_match_oracle(cells, passivate, bands):
    """8, 24 and 200 atoms; FP64 at 1e-12, FP32 blocks at 2e-6 (the bounds of
    the other product tests); three columns as single products."""
    M = _models.gaas_box(cells=cells, strain_nm=0.02, seed=41, alloy=True, phi=True,
                         passivate=passivate, band=BANDS[bands])
    ref = oracle.assemble(M.arrays())
    for prec, tol in ((native.PREC_FP64, 1e-12), (native.PREC_FP32, 2e-6)):
        H = Hamiltonian(M, layout=native.LAYOUT_BLOCKS, precision=prec)
        print(M.n_atoms, bands, prec, flush=True)
        X = _models.random_vectors(H.n, 3, seed=42)
        Y = H.hV(X, 0.6)
        for x, y in zip(X, Y):
            w = ref.hv(x, 0.6)
            assert np.linalg.norm(y - w) <= tol * np.linalg.norm(w)
            assert np.array_equal(H.hv(x, 0.6), y)


@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 2, 1)])
def test_lanczos_on_rows(cells):
    """alpha, beta of 12 steps to 1e-9 eV (see the one-launch step's test)."""
    H = Hamiltonian(_models.gaas_box(cells=cells, strain_nm=0.01, seed=43),
                    layout=native.LAYOUT_BLOCKS)
    q = _models.random_vectors(H.n, 1, seed=44)[0]
    q /= np.linalg.norm(q)
    a, b = device_tridiagonal(H, q, 12)
    ar, br = tridiagonal(H, q, 12)
    assert np.abs(a - ar).max() < 1e-9 and np.abs(b - br).max() < 1e-9
