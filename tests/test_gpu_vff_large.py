"""The relaxation where a workgroup takes more than one part of the atoms (the
gradient above 65,536 atoms, the step above 131,072): its sums against numpy's
and the oracle's energy, a short descent against the one written out on the
host."""
import numpy as np
import pytest

import _models
from nemo3d_amd import vff
from oracle import vff_oracle
from test_gpu_vff_descent import descent

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,boundary", [("VFF_keating", "FixSurfaceAll"),
                                            ("VFF_keating_strained", "AllFree")])
def test_sums_and_descent(model, boundary):
    """Sums of half a million terms of either order: 1e-12 relative for the
    energy (positive terms; n eps / 2 = 6e-11 at the very worst, sqrt(n) eps =
    2e-13 for errors of random sign), 1e-9 of the largest displacement after
    three steps of the line search."""
    M = _models.gaas_box(cells=(26, 26, 25), strain_nm=0.01, seed=37, alloy=True)
    print("atoms", M.n_atoms, flush=True)
    assert M.n_atoms > 131072
    kw = dict(model=model, boundary=boundary)
    al, be, a0 = vff.keating_tables(M)
    extra = {}
    if model == "VFF_keating_strained":
        extra = dict(zip(("aa", "ba", "ca"), vff.anharmonic_tables(M)), model=model)
    e_ref = vff_oracle.energy(M.structure, M.species, al, be, a0, **extra)
    e0, g = vff.energy_grad(M, **kw)
    print("energy", e0, "oracle", e_ref, flush=True)
    assert abs(e0 - e_ref) <= 1e-12 * e_ref
    u, it, _, e, g0, gn = descent(M, 3, 1e-6, **kw)
    info = vff.relax(M, max_iter=3, gtol=1e-6, **kw)
    assert info["iterations"] == it == 3
    assert abs(info["energy0"] - e_ref) <= 1e-12 * e_ref
    assert abs(info["grad0"] - np.linalg.norm(g)) <= 1e-12 * np.linalg.norm(g)
    assert np.abs(M.structure.disp - u).max() <= 1e-9 * np.abs(u).max()
    for k, v in (("energy", e), ("grad0", g0), ("grad", gn)):
        assert abs(info[k] - v) <= 1e-8 * abs(v), k
