"""Blocks of atoms of the SK and matrix-free products (64 own, 64 neighbouring
atoms, 176 bonds at most, cubes of 2 x 2 x 2 cells): ragged boxes, one cell,
open surfaces, one to several columns, against the oracle; and the Lanczos
step of one launch, whose beta is a difference of sums."""
import numpy as np
import pytest

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import eigensolve_lanczos
from oracle import oracle

pytestmark = pytest.mark.gpu

LAYOUTS = {"sk": native.LAYOUT_SK, "mf": native.LAYOUT_MATRIX_FREE}
SHAPES = {
    "one_cell": dict(cells=(1, 1, 1), seed=1),
    "one_cell_open": dict(cells=(1, 1, 1), seed=2, passivate=False),
    "wire": dict(cells=(5, 1, 1), strain_nm=0.02, seed=3),
    "sheet": dict(cells=(1, 3, 4), strain_nm=0.02, seed=4, phi=True),
    "odd": dict(cells=(3, 3, 3), strain_nm=0.015, seed=5, alloy=True, phi=True),
}


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_blocks_match_oracle(shape, layout):
    """FP64 at 1e-12, FP32 products at 3e-7 (the bounds of the other product
    tests), 1, 2 and 9 columns; the columns of one launch and a single
    product agree to rounding."""
    M = _models.gaas_box(**SHAPES[shape])
    ref = oracle.assemble(M.arrays())
    for prec, tol in ((native.PREC_FP64, 1e-12), (native.PREC_FP32, 3e-7)):
        print(shape, layout, prec, flush=True)
        H = Hamiltonian(M, layout=LAYOUTS[layout], precision=prec)
        X = _models.random_vectors(H.n, 9, seed=6)
        want = [ref.hv(x, 0.4) for x in X]
        for k in (1, 2, 9):
            Y = H.hV(X[:k], 0.4)
            for y, w in zip(Y, want):
                assert np.linalg.norm(y - w) <= tol * np.linalg.norm(w)
        y = H.hv(X[0], 0.4)
        assert np.linalg.norm(y - Y[0]) <= (1e-14 if tol < 1e-10 else 1e-6) * np.linalg.norm(y)


def tridiagonal(H, q, steps):
    """The same recurrence with host vectors and the device's product."""
    alpha, beta, prev, b = [], [], np.zeros_like(q), 0.0
    for _ in range(steps):
        u = H.hv(q) - b * prev
        a = np.vdot(q, u).real
        r = u - a * q
        b = np.linalg.norm(r)
        alpha.append(a)
        beta.append(b)
        prev, q = q, r / b
    return np.array(alpha), np.array(beta)


def device_tridiagonal(H, q, steps):
    r = eigensolve_lanczos(H, num_vb=0, num_cb=1, erange_cb=(1e3, 1e3 + 1),
                           max_iter=steps + 1, start_iter=10 * steps, start_vector=q,
                           want_vectors=False, return_tridiag=True)
    return r["alpha"][:steps], r["beta"][:steps]


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 2, 3)])
def test_one_launch_step_matches_recurrence(cells, layout):
    """alpha, beta of 12 steps: each step adds a few roundings of |H| (below
    40 eV) and amplifies earlier ones by |H| / beta (below 10): 1e-11 holds
    12 steps from 1e-15 with a wide margin only if nothing but rounding
    differs; 1e-9 eV is asked."""
    H = Hamiltonian(_models.gaas_box(cells=cells, strain_nm=0.01, seed=8),
                    layout=LAYOUTS[layout])
    q = _models.random_vectors(H.n, 1, seed=9)[0]
    q /= np.linalg.norm(q)
    a, b = device_tridiagonal(H, q, 12)
    ar, br = tridiagonal(H, q, 12)
    assert np.abs(a - ar).max() < 1e-9 and np.abs(b - br).max() < 1e-9


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
def test_start_near_an_eigenvector(layout):
    """A start vector 1e-7 off an eigenvector: beta_0 is about 1e-6, and
    |u|^2 - alpha^2 alone would leave it 1e-15 / 1e-6 off.  The run falls back
    to |r|^2 and keeps it to the product's rounding (1e-15 x 40 eV, a dozen of
    them: 1e-12); the eigenvalue found from it is the oracle's to 1e-9."""
    M = _models.gaas_box(cells=(2, 1, 1), strain_nm=0.01, seed=10)
    w, Z = np.linalg.eigh(oracle.assemble(M.arrays()).dense())
    H = Hamiltonian(M, layout=LAYOUTS[layout])
    i = int(np.argmin(np.abs(w - 1.0)))
    p = _models.random_vectors(H.n, 1, seed=11)[0]
    q = Z[:, i] + 1e-7 * p / np.linalg.norm(p)
    q /= np.linalg.norm(q)
    a, b = device_tridiagonal(H, q, 3)
    r = H.hv(q)
    ar = np.vdot(q, r).real
    br = np.linalg.norm(r - ar * q)
    print("alpha_0 %.3f beta_0 %.3e" % (ar, br), flush=True)
    assert br < 1e-5
    assert abs(a[0] - ar) < 1e-12 and abs(b[0] - br) < 1e-12
    assert abs(a[0] - w[i]) < 1e-9
