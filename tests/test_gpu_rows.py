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


@pytest.mark.parametrize("precision", [native.PREC_FP64, native.PREC_FP32])
@pytest.mark.parametrize("layout", [native.LAYOUT_BLOCKS, native.LAYOUT_SK,
                                    native.LAYOUT_MATRIX_FREE])
def test_columns_shared_out(layout, precision):
    """11 columns of a box whose blocks do not fill the chip: the workgroups
    take two or three columns each, the last ones fewer; the products are
    those of a column per workgroup (the same operations) and of all columns
    in one, padding untouched."""
    M = _models.gaas_box(cells=(9, 8, 6), strain_nm=0.01, seed=3)
    print("atoms", M.n_atoms, layout, precision, flush=True)
    H = Hamiltonian(M, layout=layout, precision=precision)
    n, ld, k = H.n, H.n + 8, 11
    X = np.zeros((k, ld), dtype=np.complex128)
    X[:, :n] = _models.random_vectors(n, k, seed=4)
    dX = native.DeviceArray.from_host(H, X)
    out = []
    for mode in (0, 1, -1):
        H.set(native.SET_BLOCK_HV, mode)
        dY = native.DeviceArray.from_host(H, np.full((k, ld), 2.0 + 5.0j))
        native.check(native.load().nh_hV(H.ctx, 0.3, native.ptr(dX), native.ptr(dY),
                                         k, ld, native.PTR_DEVICE))
        out.append(dY.download())
    assert np.all(out[2][:, n:] == 2.0 + 5.0j)
    for Y in out[1:]:
        err = np.linalg.norm(Y[:, :n] - out[0][:, :n]) / np.linalg.norm(out[0][:, :n])
        assert err <= (1e-15 if precision == native.PREC_FP64 else 1e-7)
