"""The relaxation's descent on the device: the same descent written out on the
host with the library's energy and gradient, over atom counts that are no
multiple of a workgroup's 64, a batch's end inside the descent, and limits of
0 and 1 steps."""
import numpy as np
import pytest

import _models
from nemo3d_amd import vff

pytestmark = pytest.mark.gpu


def descent(M, max_iter, gtol, **kw):
    """Polak-Ribiere+ with the secant line search (eight points at most)."""
    u = np.array(M.structure.disp)
    e0, g = vff.energy_grad(M, u, **kw)
    gg = (g * g).sum()
    g0, d, step, it = np.sqrt(gg), -g, 1e-4, 0
    while it < max_iter and np.sqrt(gg) > gtol:
        dg0 = (d * g).sum()
        if dg0 >= 0.0:
            d, dg0 = -g, -gg
        t0, f0, t1 = 0.0, dg0, step
        for _ in range(8):
            f1 = (vff.energy_grad(M, u + t1 * d, **kw)[1] * d).sum()
            if abs(f1) <= 1e-3 * abs(dg0):
                break
            tn = 2.0 * t1 if f1 < 0.0 and f1 <= f0 else t1 - f1 * (t1 - t0) / (f1 - f0)
            if not tn > 0.0 or not np.isfinite(tn):
                tn = 0.5 * t1
            t0, f0, t1 = t1, f1, tn
        step = t1
        u = u + t1 * d
        gt = vff.energy_grad(M, u, **kw)[1]
        bet = max(0.0, ((gt * gt).sum() - (gt * g).sum()) / gg)
        g, gg = gt, (gt * gt).sum()
        d = -g + bet * d
        it += 1
    return u, it, e0, vff.energy_grad(M, u, **kw)[0], g0, np.sqrt(gg)


@pytest.mark.parametrize("cells,max_iter,model,boundary", [
    ((1, 1, 1), 3, "VFF_keating", "AllFree"),
    ((2, 1, 1), 0, "VFF_keating", "FixSurfaceAll"),
    ((3, 2, 1), 1, "VFF_keating_strained", "AllFree"),
    ((3, 3, 2), 12, "VFF_keating", "FixSurfaceAll"),
    ((3, 3, 3), 9, "VFF_keating_strained", "FixSurfaceAll"),
])
def test_descent_matches_host(cells, max_iter, model, boundary):
    """Displacements to 1e-9 of the largest: sums in another order (1e-16 each)
    pass through at most 12 steps of the line search."""
    M = _models.gaas_box(cells=cells, strain_nm=0.01, seed=31, alloy=True)
    kw = dict(model=model, boundary=boundary)
    u, it, e0, e, g0, gn = descent(M, max_iter, 1e-6, **kw)
    info = vff.relax(M, max_iter=max_iter, gtol=1e-6, **kw)
    print(cells, model, "steps", it, "energy", e0, "->", e, flush=True)
    assert info["iterations"] == it
    assert np.abs(M.structure.disp - u).max() <= 1e-9 * np.abs(u).max()
    for k, v in (("energy0", e0), ("energy", e), ("grad0", g0), ("grad", gn)):
        assert abs(info[k] - v) <= 1e-8 * abs(v), k
