"""Weight gradients where an input is infinite or not a number at points that no
gradient reaches: those points do not count."""
import numpy as np
import pytest

import _models
from nemo3d_amd import learned
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import cnn_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("dims,c_in,layers,c_out,point", [
    ((7, 9, 13), 5, 1, 7, (3, 4, 6)),
    ((7, 9, 13), 5, 1, 7, (0, 8, 12)),
    ((6, 7, 30), 33, 2, 66, (5, 3, 15)),
    ((1, 1, 9), 16, 1, 3, (0, 0, 8)),
])
def test_unreached_points(dims, c_in, layers, c_out, point, value):
    """The gradient of the outputs is zero within `layers` of the point, so the
    parameters' gradient is that of the features with a zero there (bound of
    the network's other tests)."""
    H = Hamiltonian(_models.si_box(cells=(1, 1, 1)), layout=None)
    rng = np.random.default_rng(17)
    P = int(np.prod(dims))
    shape = dict(c_in=c_in, width=32, layers=layers, c_out=c_out)
    net = learned.CNN(H, c_in, 32, layers, c_out, seed=3)
    p = net.get_params().astype(np.float64)
    feats = rng.normal(size=(*dims, c_in)).astype(np.float32)
    dout = rng.normal(size=(*dims, c_out)).astype(np.float32)
    near = tuple(slice(max(c - layers, 0), c + layers + 1) for c in point)
    dout[near] = 0.0
    feats[point] = 0.0
    # no gradient through gates within the rounding of their sums
    _, cache, _ = cnn_oracle.forward(p, feats.reshape(P, -1), dims, keep=True, **shape)
    assert min(np.abs(pre).min() for _, pre in cache) > 1e-7
    want = cnn_oracle.backward(p, feats.reshape(P, -1), dims, dout=dout.reshape(P, -1), **shape)
    feats[point] = value
    got = net.grad(feats.reshape(P, -1), dims, dout.reshape(P, -1))
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max()
