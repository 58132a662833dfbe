"""Grids with more planes or lines than a launch has rows (65,535)."""
import numpy as np
import pytest

import _models
from nemo3d_amd import learned
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import cnn_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(65535, 1, 1), (65537, 1, 2), (140001, 1, 1), (1, 530000, 1),
                                  (1, 1, 70000)])
def test_forward_and_gradient(dims):
    """Bounds of the network's other tests; no gradient where a gate is within
    the rounding of its sum."""
    H = Hamiltonian(_models.si_box(cells=(1, 1, 1)), layout=None)
    rng = np.random.default_rng(19)
    P = int(np.prod(dims))
    shape = dict(c_in=2, width=32, layers=1, c_out=3)
    net = learned.CNN(H, 2, 32, 1, 3, seed=4)
    p = net.get_params().astype(np.float64)
    feats = rng.normal(size=(P, 2)).astype(np.float32)
    want, cache, _ = cnn_oracle.forward(p, feats, dims, keep=True, **shape)
    got = net.forward(feats, dims)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    dout = rng.normal(size=(P, 3)).astype(np.float32)
    dout[(np.abs(cache[0][1]) < 5e-6).any(axis=-1).ravel()] = 0.0
    g = cnn_oracle.backward(p, feats, dims, dout=dout, **shape)
    assert np.abs(net.grad(feats, dims, dout) - g).max() <= 1e-4 * np.abs(g).max()
