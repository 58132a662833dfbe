"""The convergence check of the Lanczos runs on the device: eigenvalues of a
given tridiagonal (a run continued from saved alpha, beta does nothing else)
against LAPACK, and which of them count as converged."""
import numpy as np
import pytest
from scipy.linalg import eigh_tridiagonal

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import eigensolve_lanczos

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    return Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=native.LAYOUT_SK)


def matrix(m, kind):
    rng = np.random.default_rng(m)
    a = rng.uniform(-5.0, 15.0, m)
    b = rng.uniform(3.0, 10.0, m)
    if kind == "graded":  # off-diagonals fall towards the end: many converged ones
        b *= np.logspace(0, -9, m)
        b = np.maximum(b, 1e-2 * np.abs(a))
    elif kind == "split":  # nearly decoupled blocks
        b[m // 3::7] = 0.2
    return a, b


@pytest.mark.parametrize("kind", ["random", "graded", "split"])
@pytest.mark.parametrize("m", [3, 7, 8, 9, 63, 64, 65, 129, 1000, 4099])
def test_windows_match_lapack(H, m, kind):
    """All eigenvalues of the two windows that a run may report (25 + 24 per
    window, the nearest to the gap), to 1e-12 (bisection to 1e-13 and rounding
    of |T| < 40), if their last two components are below the tolerance; none
    that is well above it."""
    a, b = matrix(m, kind)
    w, z = eigh_tridiagonal(a, b[:m - 1])
    tol = 1e-6
    vb, cb = (-30.0, 4.0), (6.0, 60.0)
    r = eigensolve_lanczos(H, num_vb=25, num_cb=25, erange_vb=vb, erange_cb=cb, tol=tol,
                           max_iter=m + 1, start_iter=10 * m, want_vectors=False, capacity=64,
                           restore=(a, b))
    got = np.sort(r["eigenvalues"])
    tail = np.maximum(np.abs(z[-1]), np.abs(z[-2]))
    inv = np.nonzero((w > vb[0]) & (w < vb[1]))[0][-49:]
    inc = np.nonzero((w > cb[0]) & (w < cb[1]))[0][:49]
    sure, maybe = [], []
    for idx, near in ((inv[::-1], True), (inc, False)):
        for i in idx:
            if tail[i] < 2 * tol:
                maybe.append(w[i])
            if tail[i] < 0.5 * tol:
                sure.append(w[i])
    print(m, kind, "found", got.size, "sure", len(sure), "possible", len(maybe), flush=True)
    sure, maybe = np.array(sure), np.array(maybe)
    for g in got:
        assert np.abs(maybe - g).min() < 1e-12
    # values closer than the reference's resolution (100 tol, relative or
    # absolute) count once: every sure one has a reported value that near it,
    # unless more than 25 of its window are reported
    for lo, hi in (vb, cb):
        s = sure[(sure > lo) & (sure < hi)] if sure.size else sure
        g = got[(got > lo) & (got < hi)]
        if g.size < 25:
            for x in s:
                assert g.size and np.abs(g - x).min() < 100 * tol * max(abs(x), 1.0) + 1e-12
