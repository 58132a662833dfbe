"""The work a user of the framework has it do, as cases that can be timed.

A case is a dict of plain values; `prepare` makes what a program holds
before the call (the structure's Hamiltonian on the device, vectors, a
network), `run` makes one pass through the public entry points, `work` says
what that pass cannot do without and `exact` gives its outputs in 64 bits
from plain torch.  Kinds:

  hv        Y = (H - shift) X, one or several device vectors
  lanczos   a fixed number of Lanczos steps: the tridiagonal
  solve     a whole eigensolve, eigenvectors included
  assemble  H built anew (after a relaxation) and applied once
  relax     a bounded Keating relaxation of the positions
  start     the learned start block of a structure (inference)
  train     one training step of the network on one structure

Structures are In_x Ga_(1-x) As dome dots on a wetting layer in a GaAs box,
or a plain GaAs box (base 0), with dangling-bond passivation.  Their
positions are the ideal ones displaced by the elastic field of a misfitting
sphere plus a random part, which gives every bond its own strain without
the time of a relaxation; the seed draws the alloy, the random part and the
vectors.

A solve returns its eigenvalues: Rayleigh quotients of the eigenvectors,
which stay on the device.  The vectors themselves are no comparable output
(a level is a Kramers pair, any combination of the two is an answer, and
whatever is within the tolerance is one too).
"""
import copy
import functools
import math
import os

import numpy as np
import torch

import nemo3d_amd
from nemo3d_amd import learned, materials, model, native, structure, vff, warmstart
from nemo3d_amd.hamiltonian import Hamiltonian
from nemo3d_amd.solvers import eigensolve_lanczos, eigensolve_mixed

LAYOUT = {"blocks": native.LAYOUT_BLOCKS, "sk": native.LAYOUT_SK,
          "matrix_free": native.LAYOUT_MATRIX_FREE}
BANDS = {10: materials.BANDS_10_NOSPIN, 20: materials.BANDS_20_SPIN}
WEIGHTS = os.path.join(os.path.dirname(nemo3d_amd.__file__), "data", "warmstart.npz")
HNORM = 40.0  # spectral radius of H, eV


def _dot(kind, bx, by, bz, base=0.0, height=0.0, x=1.0, bands=20, layout="sk", **more):
    return dict(kind=kind, bx=bx, by=by, bz=bz, base=base, height=height, x=x,
                bands=bands, layout=layout, **more)


def listed():
    return [
        # the plain method's small example: a 10 x 10 x 10-cell GaAs box,
        # spinless (8,000 atoms); one product inside a caller's own solver
        dict(_dot("hv", 5.66, 5.66, 5.66, bands=10, cols=1, shift=0.0), name="hv_box8k"),
        # the same at the benchmark's dot (786,520 atoms, N = 15.7M)
        dict(_dot("hv", 30.0, 30.0, 20.0, 20.0, 5.0, cols=1, shift=0.7), name="hv_dot786k"),
        # the Hamiltonian class's default layout on a dot of a few nm
        dict(_dot("hv", 15.3, 15.3, 10.2, 9.0, 3.0, 0.8, layout="blocks", cols=1, shift=0.7),
             name="hv_blocks"),
        # block products of the block solvers and of the refinement, on a dot
        # of the training set's box, matrix-free
        dict(_dot("hv", 24.0, 24.0, 16.0, 18.0, 5.0, 0.8, layout="matrix_free", cols=8,
                  shift=0.7), name="hv_8columns"),
        # the eigenvalue pass of the plain solver at the benchmark's dot
        dict(_dot("lanczos", 30.0, 30.0, 20.0, 20.0, 5.0, steps=100), name="lanczos_dot786k"),
        # the same, matrix-free, at the largest shape that is run on one GPU
        # (4.3M atoms, N = 86.7M)
        dict(_dot("lanczos", 50.0, 50.0, 40.0, 30.0, 8.0, 0.7, layout="matrix_free", steps=24),
             name="lanczos_4m"),
        # a test deck's dot (about 4,000 atoms): one level on each side of
        # the gap, FP64; latency and launches count
        dict(_dot("solve", 5.1, 5.1, 3.4, 3.4, 1.7, 0.8, form="plain"), name="solve_small"),
        # the headline form (FP32 products and vectors, FP64 refinement) on a
        # dot of 170,000 atoms
        dict(_dot("solve", 18.1, 18.1, 12.1, 11.0, 3.4, 0.8, form="mixed"), name="solve_mixed"),
        # H rebuilt for new positions, training-set dot
        dict(_dot("assemble", 24.0, 24.0, 16.0, 18.0, 5.0, 0.8), name="assemble"),
        # the positions of a new structure: the first 40 steps of the descent
        dict(_dot("relax", 15.3, 15.3, 10.2, 9.0, 3.0, 0.8, steps=40), name="relax"),
        # the learned start of the benchmark's dot
        dict(_dot("start", 30.0, 30.0, 20.0, 20.0, 5.0, 0.9), name="cnn_start"),
        # one step of training on one structure of the training set
        dict(_dot("train", 24.0, 24.0, 16.0, 18.0, 5.0, 0.8), name="cnn_train"),
    ]


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "lanczos", "lanczos", "solve", "assemble", "relax",
                       "start", "train"])
    lo, hi = {"hv": (4.0, 29.0), "lanczos": (5.0, 28.0), "solve": (4.6, 12.0),
              "assemble": (5.0, 24.0), "relax": (5.0, 15.0), "start": (8.0, 29.0),
              "train": (8.0, 23.0)}[kind]
    bx = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    by = bx * rng.uniform(0.8, 1.0)
    bz = bx * rng.uniform(0.6, 0.67)
    base = by * rng.uniform(0.55, 0.7)
    c = _dot(kind, round(bx, 3), round(by, 3), round(bz, 3), round(base, 3),
             round(bz * rng.uniform(0.25, 0.35), 3), round(rng.uniform(0.6, 0.95), 3))
    if kind == "hv":
        c["bands"] = rng.choice([10, 20, 20, 20])
        c["layout"] = rng.choice(["sk", "sk", "matrix_free", "blocks"])
        c["cols"] = rng.choice([1, 1, 1, 2, 3, 4, 5, 8]) if bx < 24.0 else 1
        c["shift"] = round(rng.uniform(-0.5, 1.5), 3)
    elif kind == "lanczos":
        c["bands"] = rng.choice([10, 20, 20])
        c["layout"] = rng.choice(["sk", "sk", "matrix_free", "blocks"]) if bx < 20.0 else "sk"
        c["steps"] = rng.randrange(40, 101)
    elif kind == "solve":
        c["form"] = rng.choice(["plain", "mixed"]) if bx < 8.0 else "mixed"
        c["layout"] = rng.choice(["sk", "sk", "matrix_free"])
    elif kind == "assemble":
        c["layout"] = rng.choice(["sk", "matrix_free", "blocks"]) if bx < 18.0 else "sk"
    elif kind == "relax":
        c["steps"] = rng.randrange(20, 41)
    return c


# ---- structures ------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _geometry(bx, by, bz, base, height):
    """The structure with every dot cation In; what the seed does not touch."""
    a = warmstart.A_GAAS
    if base == 0.0:
        cells = np.maximum(1, np.floor(np.array([bx, by, bz]) / a + 1e-9)).astype(int)
        s = structure.binary_box(tuple(cells), "Ga", "As", (a, a, a))
        s.elements.append("In")
        return s
    return structure.dot_structure((bx, by, bz), (a, a, a), base_nm=base, height_nm=height,
                                   wl_ml=1)


def _model(case, seed, displaced=True):
    g = _geometry(*(float(case[k]) for k in ("bx", "by", "bz", "base", "height")))
    s = copy.copy(g)
    rng = np.random.default_rng(seed)
    if case["x"] < 1.0:
        swap = (g.species == 2) & (rng.random(g.n_atoms) >= case["x"])
        s.species = np.where(swap, 0, g.species).astype(np.int32)
    if displaced:
        s.disp = rng.standard_normal((g.n_atoms, 3)) * 0.002
        dot = np.nonzero(g.species == 2)[0]
        if dot.size:
            p = g.positions(strained=False)
            d = p - p[dot].mean(axis=0)
            # sphere of the dome's volume; the field falls off as 1 / r^2
            h, r = case["height"], 0.5 * case["base"]
            R = (h * (3.0 * r * r + h * h) / 8.0) ** (1.0 / 3.0)
            q = np.maximum(np.sqrt((d * d).sum(axis=1)) / R, 1.0)
            s.disp += 0.03 * case["x"] * d / (q ** 3)[:, None]
    else:
        s.disp = np.zeros((g.n_atoms, 3))
    return model.TBModel(s, warmstart.COMPOUNDS, BANDS[case["bands"]], passivate=True,
                         db_shift=30.0)


class _Memory:
    """A native.DeviceArray as torch sees it (no copy)."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str,
                                         "data": (a.ptr.value, False), "version": 2}


def _fill(t, seed):
    """Normalised random entries, from the seed."""
    gen = torch.Generator(device=t.device).manual_seed(int(seed) + 1)
    r = torch.view_as_real(t)
    r.copy_(torch.randn(r.shape, generator=gen, device=t.device, dtype=torch.float64))
    t /= torch.linalg.vector_norm(t, dim=-1, keepdim=True)
    return t


def _vectors(H, shape):
    """Device vectors of the library and torch's view of them."""
    a = native.DeviceArray(H, shape)
    return a, torch.as_tensor(_Memory(a), device="cuda")


def _fill_targets(t, M, seed):
    """Eight confined states and their Kramers partners, as a training step
    gets them from the solver: random amplitudes under envelopes on the dot."""
    _fill(t, seed)
    p = M.structure.positions()
    dot = M.structure.dot_region
    r2 = torch.as_tensor(((p - p[dot].mean(axis=0)) ** 2).sum(axis=1), device=t.device)
    size = 0.3 * float(np.ptp(p[dot][:, 0]))
    for e in range(8):
        v = t[2 * e].reshape(-1, 2, 10)
        v *= torch.exp(-r2 / (size * (1.0 + 0.1 * e)) ** 2)[:, None, None]
        v /= torch.linalg.vector_norm(v)
        w = t[2 * e + 1].reshape(-1, 2, 10)
        w[:, 0] = -v[:, 1].conj()
        w[:, 1] = v[:, 0].conj()
    return t


# ---- the four functions ----------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "relax":
        s["model"] = _model(case, seed, displaced=False)
        return s
    M = s["model"] = _model(case, seed)
    if kind in ("start", "train"):
        H = s["H"] = Hamiltonian(M, layout=None)
        s["inputs"] = warmstart.structure_inputs(H)
        s["net"], _ = warmstart.load(H, WEIGHTS)
        if kind == "train":
            s["targets"], view = _vectors(H, (16, H.n))
            _fill_targets(view, M, seed)
            s["cluster"] = np.repeat(np.arange(8), 2).astype(np.int32)
            s["out_cluster"] = np.arange(8, dtype=np.int32)
    else:
        H = s["H"] = Hamiltonian(M, layout=LAYOUT[case["layout"]])
        if kind in ("hv", "assemble"):
            cols = case.get("cols", 1)
            shape = (H.n,) if cols == 1 else (cols, H.n)
            s["x"], view = _vectors(H, shape)
            _fill(view, seed)
            s["y"], s["y_view"] = _vectors(H, shape)
        elif kind == "lanczos":
            s["start"], view = _vectors(H, (H.n,))
            _fill(view, seed)
    torch.cuda.synchronize()
    return s


# the valence window ends and the conduction window begins inside the gap
WINDOWS = dict(erange_vb=(-0.4, 0.8), erange_cb=(1.25, 2.6))


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "hv":
        s["H"].hV(s["x"], case["shift"], out=s["y"])
        return s["y_view"]
    if kind == "assemble":
        s["H"].build(LAYOUT[case["layout"]])
        s["H"].hv(s["x"], out=s["y"])
        return s["y_view"]
    if kind == "lanczos":
        # as a run whose tridiagonal is saved for later: no level is asked
        # for before the last step
        r = eigensolve_lanczos(s["H"], num_vb=0, num_cb=1, erange_cb=(1e3, 1e3 + 1.0),
                               max_iter=case["steps"] + 1, start_iter=case["steps"] + 1,
                               start_vector=s["start"], want_vectors=False,
                               return_tridiag=True)
        return {"alpha": r["alpha"], "beta": r["beta"]}
    if kind == "solve":
        if case["form"] == "mixed":
            r = eigensolve_mixed(s["H"], num_vb=1, num_cb=1, tol=1e-8, tol32=3e-8, hnorm=HNORM,
                                 skip=25, stop_rule="nearest", **WINDOWS)
        else:
            r = eigensolve_lanczos(s["H"], num_vb=1, num_cb=1, tol=1e-8, max_iter=30000,
                                   skip=25, stop_rule="nearest", **WINDOWS)
        return {"eigenvalues": r["eigenvalues"]}
    if kind == "relax":
        M = s["model"]
        M.structure.disp = np.zeros((M.n_atoms, 3))
        info = vff.relax(M, max_iter=case["steps"])
        return {"disp": M.structure.disp, "energy": info["energy"]}
    if kind == "start":
        b = warmstart.start_block(s["net"], s["H"], inputs=s["inputs"], device=True)
        return torch.as_tensor(_Memory(b), device="cuda")
    g, f = s["inputs"]
    loss, grad = s["net"].train_step(f, g, s["targets"], s["cluster"], s["out_cluster"], 2e-3,
                                     want_grad=True)
    return {"loss": loss, "grad": grad, "params": s["net"].get_params()}


def _atoms(case):
    """Atoms and bonds (every atom of the box has up to four)."""
    s = _geometry(*(float(case[k]) for k in ("bx", "by", "bz", "base", "height")))
    return s.n_atoms, int((s.nbr >= 0).sum()) // 2, s


def work(case):
    """Bytes: every stored value of H once, the vectors the operation reads
    and writes once.  Operations: the bonds' 10 x 10 real blocks on complex
    vectors, the onsite terms, and, where H is stored as two-centre
    integrals or positions, the block of each bond (about 350)."""
    kind = case["kind"]
    A, nbonds, s = _atoms(case)
    nsp = case["bands"] // 10
    n = A * case["bands"]
    if case["layout"] == "blocks":
        matrix, rebuild = A * (144 + 16) + 2 * nbonds * 800, 0
    elif case["layout"] == "sk":
        matrix, rebuild = A * (144 + 36) + nbonds * 192, 350 * nbonds
    else:
        matrix, rebuild = A * (144 + 68), 450 * nbonds
    product = rebuild + 2 * nbonds * 400 * nsp + A * 120 * nsp
    if kind in ("hv", "assemble"):
        cols = case.get("cols", 1)
        b, f = matrix + 2 * 16 * n * cols, rebuild + (product - rebuild) * cols
        if kind == "assemble":  # the model read, H written
            b, f = b + matrix + A * 100, f + nbonds * 1500
    elif kind == "lanczos":  # two vectors of the recurrence read, one written
        b, f = case["steps"] * (matrix + 3 * 16 * n), case["steps"] * (product + 16 * n)
    elif kind == "solve":
        # both passes; steps grow with the box's edge (1,100 at 4,000 atoms)
        steps, size = 2 * 1100 * (A / 4000.0) ** (1.0 / 3.0), 16
        if case["form"] == "mixed":
            size, matrix = 8, A * (144 + 36) + nbonds * 96
        b, f = steps * (matrix + 3 * size * n), steps * (product + 16 * n)
    elif kind == "relax":  # about four gradients a step
        b, f = 4 * case["steps"] * A * (16 + 48 + 3 * 24), 4 * case["steps"] * A * 1500
    else:
        P = learned.GridMap(s).n_points
        macs = P * (27 * 32 * (12 + 3 * 32) + 32 * 640)
        vec = 8 * n * 16
        b, f = P * 12 * 4 + vec, 2 * macs
        if kind == "train":  # forward, and the two products of the backward
            b, f = b + vec * 2, 3 * f + 8 * n * (16 * 16 + 24 * 8)
    return {"bytes": b, "flops": f}


# ---- the same in 64 bits, in plain torch -----------------------------------

_V = {  # integrals of an (anion shell, cation shell) pair: sigma, pi, delta
    ("S", "S"): (1,), ("S", "s"): (2,), ("s", "S"): (3,), ("s", "s"): (0,),
    ("S", "p"): (6,), ("s", "p"): (4,), ("p", "S"): (7,), ("p", "s"): (5,),
    ("S", "d"): (10,), ("s", "d"): (8,), ("d", "S"): (11,), ("d", "s"): (9,),
    ("p", "p"): (12, 13), ("p", "d"): (14, 16), ("d", "p"): (15, 17),
    ("d", "d"): (18, 19, 20)}
_MINUS = {("p", "S"), ("p", "s"), ("d", "p")}  # odd l: the bond seen backwards
_ROWS = {"S": (0, 1), "s": (1, 2), "p": (2, 5), "d": (5, 10)}
# strain exponent of each of the 21 integrals, Boykin pair coefficients
_ETA = [2, 1, 0, 0, 3, 3, 7, 7, 6, 6, 14, 14, 4, 5, 8, 8, 9, 9, 11, 12, 13]
_PAIR = [[18, 19, 23, 27], [20, 17, 21, 25], [24, 22, 29, 30], [28, 26, 31, 32]]


def _quadratic(dev):
    """The d orbitals xy, yz, zx, x2-y2, 3z2-r2 as unit symmetric matrices."""
    q = torch.zeros(5, 3, 3, dtype=torch.float64, device=dev)
    h = math.sqrt(0.5)
    for k, (i, j) in enumerate([(0, 1), (1, 2), (2, 0)]):
        q[k, i, j] = q[k, j, i] = h
    q[3, 0, 0], q[3, 1, 1] = h, -h
    q[4] = torch.diag(torch.tensor([-1.0, -1.0, 2.0], dtype=torch.float64)).to(dev) / math.sqrt(6.0)
    return q


def _slater_koster(d, v):
    """Blocks T[bond, anion orbital, cation orbital] for unit vectors d
    (anion to cation) and the 21 integrals v: the orbitals are resolved in a
    frame whose third axis is the bond, where only equal |m| couple."""
    dev, nb = d.device, d.shape[0]
    ref = torch.where((d[:, 2].abs() < 0.7)[:, None], torch.tensor([0., 0., 1.], dtype=d.dtype, device=dev),
                      torch.tensor([1., 0., 0.], dtype=d.dtype, device=dev))
    e1 = torch.linalg.cross(ref, d)
    e1 = e1 / torch.linalg.vector_norm(e1, dim=1, keepdim=True)
    F = torch.stack([e1, torch.linalg.cross(d, e1), d], dim=2)  # axes as columns
    q = _quadratic(dev)
    one = torch.ones(nb, 1, 1, dtype=d.dtype, device=dev)
    local = (F.unsqueeze(1) @ q.unsqueeze(0)) @ F.transpose(1, 2).contiguous().unsqueeze(1)
    D = (q.reshape(1, 5, 9) @ local.reshape(nb, 5, 9).transpose(1, 2).contiguous())
    # components: sigma; pi (x, y; zx, yz); delta
    comp = {"S": one, "s": one, "p": F[:, :, [2, 0, 1]], "d": D[:, :, [4, 2, 1, 0, 3]]}
    T = torch.zeros(nb, 10, 10, dtype=d.dtype, device=dev)
    for (a, c), k in _V.items():
        w = torch.cat([v[:, [i]] if n == 0 else v[:, [i, i]] for n, i in enumerate(k)], dim=1)
        m = w.shape[1]
        t = (comp[a][:, :, :m] * w[:, None, :]) @ comp[c][:, :, :m].transpose(1, 2).contiguous()
        T[:, _ROWS[a][0]:_ROWS[a][1], _ROWS[c][0]:_ROWS[c][1]] = -t if (a, c) in _MINUS else t
    return T


class _Operator:
    """H of a model in 64 bits."""

    def __init__(self, M):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        m = {k: torch.as_tensor(v, device=dev) if isinstance(v, np.ndarray) else v
             for k, v in M.arrays().items()}
        A, self.nsp, self.dev = m["n_atoms"], m["nb"] // 10, dev
        cat, sp, nbr = m["is_cation"].bool(), m["species"].long(), m["nbr"].long()
        self.A, self.have = A, nbr >= 0
        self.nbr = nbr.clamp(min=0)
        # bonds: (cation, its slot)
        i, slot = torch.nonzero(self.have & cat[:, None], as_tuple=True)
        j = nbr[i, slot]
        back = torch.nonzero((nbr[j] == i[:, None]))[:, 1]
        par, strn = m["parmat"][sp[i], sp[j]], m["strnmat"][sp[i], sp[j]]
        ideal = 0.25 * m["bond_q"][i, slot].double()
        r = -(ideal * m["lattice"] + m["disp"][j] - m["disp"][i])
        length = torch.linalg.vector_norm(r, dim=1)
        ratio = 0.25 * math.sqrt(3.0) * par[:, 31] / length
        v = par[:, 10:31] * ratio[:, None] ** strn[:, _ETA]
        e = torch.zeros(A, 10, dtype=torch.float64, device=dev)
        self.T = torch.zeros(A, 4, 10, 10, dtype=torch.float64, device=dev)
        shell = [0, 1, 2, 2, 2, 3, 3, 3, 3, 3]
        pair = [[_PAIR[a][c] for c in shell] for a in shell]
        ea, ec = [4, 0, 1, 1, 1, 6, 6, 6, 6, 6], [5, 2, 3, 3, 3, 7, 7, 7, 7, 7]
        for k in range(0, i.numel(), 1 << 18):
            b = slice(k, k + (1 << 18))
            T = _slater_koster(r[b] / length[b, None], v[b])
            T0 = _slater_koster(-ideal[b] / torch.linalg.vector_norm(ideal[b], dim=1, keepdim=True),
                                par[b, 10:31])
            self.T[j[b], back[b]] = T
            self.T[i[b], slot[b]] = T.transpose(1, 2)
            # diagonal corrections of Boykin et al., pair by pair
            corr = ((T0 * T0 - T * T) * strn[b, 10, None, None] /
                    (par[b][:, ea][:, :, None] + par[b][:, ec][:, None, :]) *
                    strn[b][:, torch.tensor(pair, device=dev)])
            e.index_add_(0, j[b], corr.sum(dim=2))
            e.index_add_(0, i[b], corr.sum(dim=1))
        # onsite energies, averaged over the bonds an atom has
        c_sp = torch.where(cat[:, None], sp[:, None], sp[self.nbr])
        a_sp = torch.where(cat[:, None], sp[self.nbr], sp[:, None])
        w = self.have.double() / self.have.sum(dim=1, keepdim=True)
        mean = (m["parmat"][c_sp, a_sp] * w[:, :, None]).sum(dim=1)
        shift = (m["strnmat"][c_sp, a_sp][:, :, 15:17] * w[:, :, None]).sum(dim=1)
        e += torch.where(cat[:, None], mean[:, ec] + shift[:, [0]], mean[:, ea] + shift[:, [1]])
        self.lam = torch.where(cat, mean[:, 9], mean[:, 8])
        # dangling bonds: sp3 hybrids along the missing neighbours, raised
        self.surface = torch.nonzero(~self.have.all(dim=1))[:, 0]
        hyb = 0.25 * torch.tensor([[1., 1, 1], [-1, -1, 1], [1, -1, -1], [-1, 1, -1]],
                                  dtype=torch.float64, device=dev)
        su = self.surface
        dots = (0.25 * m["bond_q"][su].double()) @ hyb.t().contiguous()  # (n, slot, hybrid)
        which = dots.abs() >= 0.15
        first = torch.where(which.any(dim=2), which.int().argmax(dim=2), 3)
        up = torch.full((su.numel(), 4), 0.25 * m["db_shift"], dtype=torch.float64, device=dev)
        for n in range(4):
            k = torch.nonzero(self.have[su, n])[:, 0]
            up[k, first[k, n]] = 0.0
        sign = torch.where(dots[:, 3].gather(1, first[:, 3:4])[:, 0] > 0, 1.0, -1.0).double()
        g = torch.tensor([[1., 1, 1, 1], [1, -1, 1, -1], [1, -1, -1, 1], [1, 1, -1, -1]],
                         dtype=torch.float64, device=dev)
        z = (up @ g.t().contiguous())  # sum; s-px, s-py, s-pz patterns
        e[su, 1:5] += z[:, [0]]
        S = torch.zeros(su.numel(), 4, 4, dtype=torch.float64, device=dev)
        for a, b, val in ((0, 1, sign * z[:, 1]), (0, 2, sign * z[:, 2]), (0, 3, sign * z[:, 3]),
                          (1, 2, z[:, 3]), (1, 3, z[:, 2]), (2, 3, z[:, 1])):
            S[:, a, b] = S[:, b, a] = val
        self.S, self.e = S, e

    def __call__(self, x, shift=0.0):
        """(H - shift) x for x (..., N) complex."""
        x0 = x.reshape(-1, self.A, self.nsp, 10)
        y = (self.e - shift)[None, :, None, :] * x0
        for k in range(x0.shape[0]):
            xk = x0[k]
            for n in range(4):
                g = xk[self.nbr[:, n]] * self.have[:, n, None, None]
                cols = torch.view_as_real(g).permute(0, 2, 1, 3).reshape(self.A, 10, -1).contiguous()
                t = torch.bmm(self.T[:, n].contiguous(), cols)
                y[k] += torch.view_as_complex(
                    t.reshape(self.A, 10, self.nsp, 2).permute(0, 2, 1, 3).contiguous())
            sp = xk[self.surface][:, :, 1:5]
            y[k, self.surface, :, 1:5] += (self.S[:, None] * sp[:, :, None, :]).sum(dim=3)
            if self.nsp == 2:  # lambda L.S on the p orbitals
                l = self.lam
                (ux, uy, uz), (dx, dy, dz) = ([xk[:, s, 2 + c] for c in range(3)] for s in (0, 1))
                for s, c, t in ((0, 0, -1j * uy + dz), (0, 1, 1j * ux - 1j * dz),
                                (0, 2, -dx + 1j * dy), (1, 0, 1j * dy - uz),
                                (1, 1, -1j * dx - 1j * uz), (1, 2, ux + 1j * uy)):
                    y[k, :, s, 2 + c] += l * t
        return y.reshape(x.shape)


def _tridiagonal(H, q, steps):
    alpha, beta = [], []
    prev, b = torch.zeros_like(q), 0.0
    q = q / torch.linalg.vector_norm(q)
    for _ in range(steps):
        w = H(q) - b * prev
        a = torch.vdot(q, w).real
        w -= a * q
        b = torch.linalg.vector_norm(w)
        prev, q = q, w / b
        alpha.append(float(a))
        beta.append(float(b))
    return {"alpha": np.array(alpha), "beta": np.array(beta)}


def _shifted(a, d, dims):
    """a (gx, gy, gz, C) seen from the point p + d, zero outside."""
    out = torch.zeros_like(a)
    src = tuple(slice(max(0, k), n + min(0, k)) for k, n in zip(d, dims))
    dst = tuple(slice(max(0, -k), n + min(0, -k)) for k, n in zip(d, dims))
    out[dst] = a[src]
    return out


class _Conv(torch.autograd.Function):
    """3 x 3 x 3 convolution on a channels-last grid, shift by shift."""

    OFF = [(k // 9 - 1, (k // 3) % 3 - 1, k % 3 - 1) for k in range(27)]

    @staticmethod
    def forward(ctx, a, w):
        ctx.save_for_backward(a, w)
        dims = a.shape[:3]
        out = torch.zeros(*dims, w.shape[0], dtype=a.dtype, device=a.device)
        for k, d in enumerate(_Conv.OFF):
            out += _shifted(a, d, dims) @ w[:, :, k].t().contiguous()
        return out

    @staticmethod
    def backward(ctx, g):
        a, w = ctx.saved_tensors
        dims = a.shape[:3]
        ga, gw = torch.zeros_like(a), torch.zeros_like(w)
        G = g.reshape(-1, g.shape[3])
        for k, d in enumerate(_Conv.OFF):
            gw[:, :, k] = G.t().contiguous() @ _shifted(a, d, dims).reshape(-1, a.shape[3])
            ga += _shifted((g @ w[:, :, k]).contiguous(), tuple(-v for v in d), dims)
        return ga, gw


def _network(case, M, params):
    """Leaves of the parameters (bf16 values) and the predicted block."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = learned.GridMap(M.structure)
    f = torch.as_tensor(learned.features(M, g), device=dev).double()
    a = f.reshape(*g.dims, -1)
    p = torch.as_tensor(params, device=dev).bfloat16().double()
    leaves, off, ci = [], 0, f.shape[1]
    for size, bias in [((32, c, 27), 32) for c in (ci, 32, 32, 32)] + [((640, 32), 640)]:
        for shape in (size, (bias,)):
            n = int(np.prod(shape))
            leaves.append(p[off:off + n].reshape(shape).clone().requires_grad_())
            off += n
    for l in range(4):
        a = torch.relu(_Conv.apply(a, leaves[2 * l]) + leaves[2 * l + 1])
    point = torch.as_tensor(g.point, device=dev).long()
    slot = torch.as_tensor(g.slot, device=dev).long()
    out = (a.reshape(g.n_points, 32) @ leaves[8].t().contiguous() + leaves[9])
    out = out.reshape(g.n_points, 8, 2, 20, 2)[point, :, slot].transpose(0, 1).contiguous()
    return leaves, torch.view_as_complex(out).reshape(8, -1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "relax"):
        return None
    M = _model(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def zeros(*shape):
        return torch.zeros(*shape, dtype=torch.complex128, device=dev)

    if kind in ("hv", "assemble"):
        cols = case.get("cols", 1)
        x = _fill(zeros(M.n) if cols == 1 else zeros(cols, M.n), seed)
        return _Operator(M)(x, case.get("shift", 0.0))
    if kind == "lanczos":
        return _tridiagonal(_Operator(M), _fill(zeros(M.n), seed), case["steps"])
    params = np.load(WEIGHTS, allow_pickle=False)["params"]
    if kind == "start":
        return _network(case, M, params)[1].detach()
    V = _fill_targets(zeros(16, M.n), M, seed)
    leaves, Y = _network(case, M, params)
    C = V.conj() @ Y.t()
    loss = sum(1.0 - (C[2 * e:2 * e + 2, e].abs() ** 2).sum() / (Y[e].abs() ** 2).sum()
               for e in range(8)) / 8.0
    loss.backward()
    grad = torch.cat([l.grad.reshape(-1) for l in leaves])
    # Adam's first step from the 32-bit weights
    new = torch.as_tensor(params, device=grad.device).double() - 2e-3 * grad / (grad.abs() + 1e-8)
    return {"loss": float(loss.detach()), "grad": grad.cpu().numpy(), "params": new.cpu().numpy()}
