"""The factored bond product (nh_sk_apply.h) compiled for the host: its errors
against the Slater-Koster table in 80 bits, beside those of a product with the
table itself in FP64 and FP32; both orientations are exact transposes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FACTORED64, FACTORED32, TABLE80, TABLE64, TABLE32 = range(5)


@pytest.fixture(scope="module")
def product(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("sk") / "sk_shim.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-mfma",
                           "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-o", so,
                           os.path.join(HERE, "native", "sk_shim.cpp")])
    lib = ctypes.CDLL(so)
    P = ctypes.c_void_p

    def run(kind, cation, d, v, x):
        y = np.zeros(10)
        lib.sk_product(kind, cation, P(d.ctypes.data), P(v.ctypes.data), P(x.ctypes.data),
                       P(y.ctypes.data))
        return y

    return run


def bonds(n, off, seed):
    """Directions `off` around (111), integrals of the size of a table's."""
    rng = np.random.default_rng(seed)
    base = np.array([-1.6, -3.7, -2.0, -1.6, 3.1, 2.9, 2.2, 1.8, -2.6, -2.9, -0.7, -2.2, 4.4,
                     -1.2, -1.7, -1.8, 1.8, 2.0, -1.1, 2.2, -2.0])
    for k in range(n):
        d = np.array([1.0, 1 - 2 * (k & 1), 1 - (k & 2)]) + off * rng.standard_normal(3)
        # FP32 directions, so that all forms have the same bond up to their own rounding
        yield (d / np.linalg.norm(d), base * (1 + 0.1 * rng.standard_normal(21)),
               rng.standard_normal(10).astype(np.float32).astype(np.float64))


@pytest.mark.parametrize("off", [0.0, 0.002, 0.03, 0.5])
def test_errors_are_those_of_the_table(product, off):
    """FP64: root mean square 4e-16 of the result (about ten roundings of 6e-17,
    with intermediate values up to twice the results).  FP32: no more than the
    table formed and applied in FP32, within the spread of such a mean over
    8,000 products (2%)."""
    e = dict.fromkeys((FACTORED64, FACTORED32, TABLE64, TABLE32), 0.0)
    size = 0.0
    for d, v, x in bonds(4000, off, 5):
        for cation in (0, 1):
            want = product(TABLE80, cation, d, v, x)
            size += (want ** 2).sum()
            for k in e:
                e[k] += ((product(k, cation, d, v, x) - want) ** 2).sum()
    e = {k: np.sqrt(s / size) for k, s in e.items()}
    print(off, e)
    assert e[FACTORED64] < 4e-16
    assert e[FACTORED32] < 1.02 * e[TABLE32]


@pytest.mark.parametrize("kind", [FACTORED64, FACTORED32])
def test_orientations_are_transposes(product, kind):
    for d, v, _ in bonds(100, 0.1, 6):
        T = [np.array([product(kind, c, d, v, np.eye(10)[i]) for i in range(10)])
             for c in (0, 1)]
        assert np.array_equal(T[0], T[1].T)
