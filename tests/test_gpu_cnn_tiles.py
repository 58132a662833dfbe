"""The network's matrix-core kernels at the edges of their tiles (up to 128
points of a plane, x segments, 16 / 32 input channels, 32 / 160 head rows, 64
gradient channels) against the FP64 oracle, with the bounds of the device
network's test: FP32 sums, 1e-5 of the largest output, 1e-4 of the largest
gradient.
A relu input within the rounding of its sum (864 terms as a random walk of
2^-24 steps on partial sums of a few units: 5e-6) may open or close its gate;
the oracle's gradient is taken with either sign of such inputs.
"""
import itertools

import numpy as np
import pytest

import _models
from nemo3d_amd import learned, materials
from nemo3d_amd.hamiltonian import Hamiltonian
from oracle import cnn_oracle

pytestmark = pytest.mark.gpu

CASES = [  # dims, c_in, layers, c_out
    ((1, 1, 1), 1, 1, 1),
    ((2, 9, 17), 13, 2, 6),
    ((5, 8, 16), 16, 2, 160),
    ((3, 7, 33), 17, 2, 163),
    ((19, 3, 5), 32, 3, 64),
    ((4, 17, 15), 33, 2, 65),
    ((2, 4, 40), 64, 1, 640),
    ((40, 2, 3), 12, 4, 161),
]


def gradients(monkeypatch, p, feats, dims, dout, shape):
    """The oracle's gradient for every choice of the undecided gates."""
    out, cache, x = cnn_oracle.forward(p, feats, dims, keep=True, **shape)
    open_ = [(l, i) for l, (_, pre) in enumerate(cache)
             for i in np.argwhere(np.abs(pre) < 5e-6)]
    assert len(open_) <= 4
    res = []
    for signs in itertools.product((1.0, -1.0), repeat=len(open_)):
        for (l, i), s in zip(open_, signs):
            cache[l][1][tuple(i)] = s * 1e-9
        with monkeypatch.context() as m:
            m.setattr(cnn_oracle, "forward", lambda *a, **k: (out, cache, x))
            res.append(cnn_oracle.backward(p, feats, dims, dout=dout, **shape))
    return res


@pytest.fixture(scope="module")
def owner():
    return Hamiltonian(_models.si_box(cells=(1, 1, 1)), layout=None)


@pytest.mark.parametrize("dims,c_in,layers,c_out", CASES)
def test_forward_and_gradient(owner, monkeypatch, dims, c_in, layers, c_out):
    print(dims, c_in, layers, c_out, flush=True)
    rng = np.random.default_rng(5)
    shape = dict(c_in=c_in, width=32, layers=layers, c_out=c_out)
    P = int(np.prod(dims))
    feats = rng.normal(size=(P, c_in)).astype(np.float32)
    dout = rng.normal(size=(P, c_out)).astype(np.float32)
    net = learned.CNN(owner, c_in, 32, layers, c_out, seed=6)
    p = net.get_params().astype(np.float64)
    ref = cnn_oracle.forward(p, feats, dims, **shape)
    assert np.abs(net.forward(feats, dims) - ref).max() <= 1e-5 * np.abs(ref).max()
    g = net.grad(feats, dims, dout)
    assert any(np.abs(g - r).max() <= 1e-4 * np.abs(r).max()
               for r in gradients(monkeypatch, p, feats, dims, dout, shape))
    assert np.array_equal(g, net.grad(feats, dims, dout))  # sums in a fixed order


@pytest.mark.parametrize("dims", [(256, 30, 4), (256, 3, 32), (128, 25, 5), (300, 6, 20)])
def test_tiles_of_other_shapes(owner, dims):
    """Grids that take narrow, wide and ragged tiles (30 x 4, 3 x 32, ...):
    two layers forward and backward.  No gradient is put in where a gate
    within the rounding of its sum could pass it on or not."""
    print(dims, flush=True)
    rng = np.random.default_rng(8)
    shape = dict(c_in=5, width=32, layers=2, c_out=3)
    P = int(np.prod(dims))
    feats = rng.normal(size=(P, 5)).astype(np.float32)
    net = learned.CNN(owner, 5, 32, 2, 3, seed=9)
    p = net.get_params().astype(np.float64)
    ref, cache, _ = cnn_oracle.forward(p, feats, dims, keep=True, **shape)
    assert np.abs(net.forward(feats, dims) - ref).max() <= 1e-5 * np.abs(ref).max()
    near = [(np.abs(pre) < 5e-6).any(axis=-1) for _, pre in cache]
    shut = near[1].copy()
    for x, y, z in np.argwhere(near[0]):
        shut[max(x - 1, 0):x + 2, max(y - 1, 0):y + 2, max(z - 1, 0):z + 2] = True
    dout = rng.normal(size=(P, 3)).astype(np.float32)
    dout[shut.ravel()] = 0.0
    r = cnn_oracle.backward(p, feats, dims, dout=dout, **shape)
    assert np.abs(net.grad(feats, dims, dout) - r).max() <= 1e-4 * np.abs(r).max()


@pytest.mark.parametrize("bands,ne,targets,device", [
    (20, 1, 1, True), (20, 3, 9, False), (20, 8, 16, True), (10, 5, 8, False), (10, 8, 16, True)])
def test_start_block_and_step(bands, ne, targets, device):
    """10 and 20 bands (2 or 4 states a block of head rows), one to sixteen
    targets on the host or on the device."""
    from nemo3d_amd import native
    kw = dict(cells=(3, 2, 1), strain_nm=0.02, seed=8)
    M = _models.gaas_box(**kw) if bands == 20 else _models.gaas_box(
        band=materials.BANDS_10_NOSPIN, **kw)
    H = Hamiltonian(M, layout=None)
    nb = H.n // M.n_atoms
    assert nb == bands
    g = learned.GridMap(M.structure)
    rng = np.random.default_rng(9)
    shape = dict(c_in=6, width=32, layers=1, c_out=ne * 4 * nb + 3)
    feats = rng.normal(size=(g.n_points, 6)).astype(np.float32)
    net = learned.CNN(H, 6, 32, 1, shape["c_out"], seed=2)
    p = net.get_params().astype(np.float64)
    Yref = cnn_oracle.map_out(cnn_oracle.forward(p, feats, g.dims, **shape), g.point, g.slot,
                              nb, ne)
    Y = net.start_block(feats, g, ne)
    assert np.abs(Y - Yref).max() <= 1e-5 * np.abs(Yref).max()
    V = rng.normal(size=(targets, H.n)) + 1j * rng.normal(size=(targets, H.n))
    V = np.linalg.qr(V.T)[0].T.copy()
    cl = (np.arange(targets) % ne).astype(np.int32)
    oc = np.arange(ne, dtype=np.int32)
    t = native.DeviceArray.from_host(H, V) if device else V
    L, grad = net.train_step(feats, g, t, cl, oc, lr=0.0, want_grad=True)
    Lref, G = cnn_oracle.subspace_loss(Yref, V, cl, oc)
    assert abs(L - Lref) <= 1e-6 * max(abs(Lref), 1.0)
    dout = cnn_oracle.map_grad(G, g.point, g.slot, nb, ne, g.n_points, shape["c_out"])
    gref = cnn_oracle.backward(p, feats, g.dims, dout=dout, **shape)
    assert np.abs(grad - gref).max() <= 1e-3 * np.abs(gref).max()
