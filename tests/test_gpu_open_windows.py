"""Energy windows with an open end: a bound far beyond the spectrum finds what the
spectrum's own bound finds."""
import numpy as np
import pytest

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import eigensolve_lanczos

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("end", [1e30, 1e39, 1e99, np.inf])
def test_open_ends(end):
    """The same tridiagonal, so the same eigenvalues to the bisection's 1e-13."""
    H = Hamiltonian(_models.gaas_box(cells=(1, 1, 1)), layout=native.LAYOUT_SK)
    rng = np.random.default_rng(3)
    m = 203
    a, b = rng.uniform(-5.0, 15.0, m), np.maximum(rng.uniform(3.0, 10.0, m) * np.logspace(0, -9, m),
                                                  1e-6)
    kw = dict(num_vb=12, num_cb=12, tol=1e-6, max_iter=m + 1, start_iter=10 * m,
              want_vectors=False, restore=(a, b))
    bound = np.abs(a).max() + 2 * b.max()
    want = eigensolve_lanczos(H, erange_vb=(-bound, 3.0), erange_cb=(6.0, bound), **kw)
    got = eigensolve_lanczos(H, erange_vb=(-end, 3.0), erange_cb=(6.0, end), **kw)
    print(end, "found", got["eigenvalues"].size, "of", want["eigenvalues"].size, flush=True)
    assert want["converged"] and got["converged"]
    assert got["eigenvalues"].size == want["eigenvalues"].size == 24
    assert np.abs(got["eigenvalues"] - want["eigenvalues"]).max() < 1e-12
