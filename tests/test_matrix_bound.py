"""Which launches of a plan have transfer matrices, and what they take (host
stage of plan construction only, no GPU)."""
import ctypes

import numpy as np
import pytest

import libcint_amd as mc
from libcint_amd.synthetic import make_molecule, subset, unique_quartets


def _matrices(m, name, q, kib=None):
    """(tasks on the matrix kernel, on the generic one, doubles of matrices, scratch)."""
    f = mc.lib()._ZN5mcint23plan_matrices_host_onlyEPKiiS1_iPKdiS1_mPl
    ip, q = ctypes.POINTER(ctypes.c_int), np.ascontiguousarray(q, np.int32)
    n = (ctypes.c_int64 * 4)()
    old = None if kib is None else mc.tune(mc.TUNE_MATRIX_KIB, kib)
    try:
        rc = f(m.atm.ctypes.data_as(ip), len(m.atm), m.bas.ctypes.data_as(ip), len(m.bas),
               m.env.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), mc.INTOR_CODES[name],
               q.ctypes.data_as(ip), ctypes.c_size_t(len(q)), n)
    finally:
        if old is not None:
            mc.tune(mc.TUNE_MATRIX_KIB, old)
    assert rc == 0
    return list(n)


@pytest.mark.parametrize("name", ["int2e_ipip1_sph", "int2e_ip1ip2_cart", "int3c2e_ip2_sph", "int2c2e_sph"])
def test_bound_takes_classes_not_plans(name):
    """A bound below what all matrices take leaves the costliest classes on the
    matrix kernel; every task keeps one of the two kernels."""
    three = "c2e" in name
    m = make_molecule("c4") if three else subset(make_molecule("c3"), 3)
    if three:
        aux = np.arange(m.aux_start, m.nbas)[::7]
        q = np.array([(i, j, k, 0) for i in range(0, m.aux_start, 9) for j in range(0, m.aux_start, 11)
                      for k in aux], np.int32)
        if name.startswith("int2c2e"):
            q[:, 0], q[:, 1] = q[:, 2], np.resize(aux, len(q))
    else:
        q = unique_quartets(m.nbas)
    on, off, size, _ = _matrices(m, name, q)
    assert on > 0 and size > 0
    last, seen = (on, size), set()
    for kib in (size // 128 + 1, size // 256, size // 512, size // 1024, 0):
        n, g, s, _ = _matrices(m, name, q, kib)
        assert n + g == on + off and s <= kib * 128
        assert (n, s) <= last
        assert (n, s) == (on, size) or g > off
        seen.add(n)
    assert (n, s) == (0, 0)
    assert len(seen) > 2, "the bound is not all or nothing"


def test_layout_does_not_depend_on_threads():
    """Long lists collect their pairs on several threads: the same matrices
    (with 0 lanes to fill the kernel of a class does not depend on its list)."""
    m = subset(make_molecule("c3"), 3)
    q = unique_quartets(m.nbas)
    long = np.tile(q, (-(-400000 // len(q)), 1))
    old = mc.tune(mc.TUNE_FILL_LANES, 0)
    try:
        a, b = _matrices(m, "int2e_ipip1_sph", q), _matrices(m, "int2e_ipip1_sph", long)
    finally:
        mc.tune(mc.TUNE_FILL_LANES, old)
    assert a[2] == b[2] and b[0] == a[0] * (len(long) // len(q))


def _one_class(ls, nprim, n):
    """n random tuples of shells of angular momenta ls with nprim primitives."""
    env, atm, bas = [0.0] * 20, [], []
    rng = np.random.default_rng(5)
    for _ in range(4):
        atm.append([6, len(env), 1, 0, 0, 0])
        env += rng.uniform(-1.5, 1.5, 3).tolist()
    shells = {}
    for l in sorted(set(ls)):
        shells[l] = np.arange(len(bas), len(bas) + 4)
        for a in range(4):
            bas.append([a, l, nprim, 1, 0, len(env), len(env) + nprim, 0])
            env += (0.3 * 2.5 ** np.arange(nprim) * rng.uniform(0.8, 1.2)).tolist() + [0.5] * nprim
    m = make_molecule("c0")
    m.atm, m.bas, m.env = np.array(atm, np.int32), np.array(bas, np.int32), np.array(env)
    q = np.zeros((n, 4), np.int32)
    for i, l in enumerate(ls):
        q[:, i] = rng.choice(shells[l], n)
    return m, q


# one class each: kind, angular momenta, primitives per shell, tuples, and
# whether the matrix kernel takes it
CLASSES = [
    ("int2e_ip1ip2_sph", (2, 2, 2, 2), 4, 600, True),    # 78 KB for four waves
    ("int2e_ip1_sph", (1, 1, 4, 3), 4, 600, True),
    ("int2e_sph", (4, 3, 4, 1), 2, 1100, True),          # four waves by the LDS
    ("int2e_ip1ip2_sph", (3, 1, 2, 3), 1, 600, True),    # 60 KB for one wave
    ("int2e_ip1ip2_sph", (3, 1, 2, 3), 4, 520, False),   # ... and many primitives
    ("int2e_cart", (4, 4, 0, 0), 1, 1100, False),        # the bra matrix outweighs the walk
    ("int2e_ipip1_sph", (2, 3, 0, 0), 1, 1100, False),
    ("int2c2e_sph", (0, 0), 1, 300, False),
    ("int2c2e_sph", (1, 1), 1, 300, True),
]


@pytest.mark.parametrize("name,ls,nprim,n,matrix", CLASSES)
def test_kernel_of_a_class(name, ls, nprim, n, matrix):
    m, q = _one_class(ls, nprim, n)
    on, off, _, _ = _matrices(m, name, q)
    assert (on, off) == ((n, 0) if matrix else (0, n))
