"""Device memory of a Lanczos run: the vectors it needs and no more."""
import ctypes

import pytest

import _models
from nemo3d_amd import native
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import eigensolve_lanczos

pytestmark = pytest.mark.gpu


def idle_bytes(H):
    free, idle = ctypes.c_int64(), ctypes.c_int64()
    native.check(native.load().nh_context_mem_info(H.ctx, ctypes.byref(free), ctypes.byref(idle)))
    return idle.value


@pytest.mark.parametrize("precision,vectors", [(native.PREC_FP64, 5), (native.PREC_FP32, 3)])
def test_eigenvalue_pass(precision, vectors):
    """r and u of two steps in the vectors' precision and the FP64 start vector,
    all in the context's pool when the run is over (besides them: partial sums,
    the tridiagonal and the check's scratch, below 1 MB + 1 MB)."""
    H = Hamiltonian(_models.gaas_box(cells=(18, 18, 18)), layout=native.LAYOUT_SK,
                    precision=precision)
    before = idle_bytes(H)
    eigensolve_lanczos(H, num_vb=1, num_cb=1, max_iter=40, start_iter=100, want_vectors=False)
    used = idle_bytes(H) - before
    print("vectors of %.1f MB: %.2f of them" % (H.n * 16e-6, used / (H.n * 16.0)), flush=True)
    assert used <= vectors * H.n * 16 + (2 << 20)


@pytest.mark.parametrize("precision", [native.PREC_FP64, native.PREC_FP32])
def test_eigenvectors_from_reused_memory(precision):
    """A run with eigenvectors: twice the same, residuals as small as the run's
    tolerance allows (tail x beta, below 1e-5 eV in FP64; FP32 products 1e-4)."""
    M = _models.gaas_box(cells=(3, 3, 3), strain_nm=0.005, seed=5)
    H = Hamiltonian(M, layout=native.LAYOUT_SK, precision=precision)
    kw = dict(num_vb=2, num_cb=2, erange_vb=(-2.0, 0.6), erange_cb=(1.0, 5.0), tol=1e-7,
              max_iter=3000, start_iter=100, skip=50)
    r = [eigensolve_lanczos(H, return_vectors=True, **kw) for _ in range(2)]
    assert r[0]["converged"] and (r[0]["vectors"] == r[1]["vectors"]).all()
    print(r[0]["eigenvalues"], r[0]["residuals"], flush=True)
    assert r[0]["residuals"].max() < (1e-5 if precision == native.PREC_FP64 else 1e-4)
