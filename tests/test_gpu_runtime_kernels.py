"""The two kernels whose class is known at run time, the matrix kernel and the
generic one, on the same lists against the CPU oracle.

A plan's runtime classes run on the matrix kernel while their transfer
matrices fit MCINT_TUNE_MATRIX_KIB; 0 leaves all of them to the generic
kernel, and a bound in between splits the classes.

Tolerance of a block: 1e-12 + 1e-10 of its largest element.  Exponents are at
most 10, so that a derivative's largest intermediate, 2a [a+1| ~ 2 sqrt(a)
times the plain integral (4a for two derivatives), is at most 40 times the
plain integral (at most about 10; 30 for aux pairs, whose blocks scale with
it), and rounding at most about 400 x 2.2e-16 x a few operations: below 1e-12.
"""
import numpy as np
import pytest

from libcint_amd.synthetic import make_molecule, random_density, subset, unique_quartets
from test_matrix_bound import CLASSES, _one_class

pytestmark = pytest.mark.gpu

KERNELS = {"matrix": None, "split": 512, "generic": 0}  # bound of the matrices, KiB


@pytest.fixture(scope="module")
def mc():
    import libcint_amd
    libcint_amd.lib()
    return libcint_amd


@pytest.fixture(scope="module")
def orc():
    import oracle
    oracle.build()
    oracle.set_root_mode(oracle.ROOTS_TABLE)
    yield oracle
    oracle.set_root_mode(oracle.ROOTS_EXACT)


class _Route:
    """Plans made inside run every class on the runtime-class kernels."""

    def __init__(self, mc, kernel):
        self.mc, self.set = mc, {mc.TUNE_GENERIC_ONLY: 1}
        if KERNELS[kernel] is not None:
            self.set[mc.TUNE_MATRIX_KIB] = KERNELS[kernel]

    def __enter__(self):
        self.old = {k: self.mc.tune(k, v) for k, v in self.set.items()}

    def __exit__(self, *_):
        for k, v in self.old.items():
            self.mc.tune(k, v)


def _molecule(config, natoms=0):
    """The workload with contractions cut to their five most diffuse primitives."""
    m = make_molecule(config)
    m = subset(m, natoms) if natoms else m
    m.bas[:, 2] = np.minimum(m.bas[:, 2], 5)
    return m


def _general(m):
    """m with a second contraction column on its first s shell."""
    s = int(np.flatnonzero((m.bas[:, 1] == 0) & (m.bas[:, 2] > 1))[0])
    n, pc = int(m.bas[s, 2]), int(m.bas[s, 6])
    m.bas[s, 3], m.bas[s, 6] = 2, len(m.env)
    m.env = np.concatenate([m.env, m.env[pc:pc + n], m.env[pc:pc + n][::-1]])
    return m


def _list(m, name, seed):
    """Every order of s, p, d (some f) shells, contracted and not, and one class
    of 33 000 quartets (several tasks per workgroup on either kernel)."""
    rng = np.random.default_rng(seed)
    ls, npr = m.bas[:, 1], m.bas[:, 2]
    orb = np.arange(m.aux_start if m.aux_start >= 0 else m.nbas)
    lo = ls[orb]
    few = np.concatenate([orb[(lo == l) & (npr[orb] == 1)][:4] for l in range(3)]
                         + [orb[(lo == l) & (npr[orb] == 5)][:2] for l in range(2)])
    q = rng.choice(few, (250, 4)).astype(np.int32)
    f = orb[lo == 3][:2]
    q[:4, 0], q[4:8, 2], q[8:10, 1] = f[0], f[-1], f[0]
    if "c2e" not in name and "ipip1" not in name and "ip1ip2" not in name:
        q[10] = f[0], f[-1], f[0], f[-1]
    long = np.empty((33000, 4), np.int32)
    for c, l in enumerate((1, 0, 1, 0)):
        long[:, c] = rng.choice(orb[(lo == l) & (npr[orb] == 1)], len(long))
    q = np.concatenate([q, long])
    if "c2e" in name:
        aux = np.arange(m.aux_start, m.nbas)
        aux = aux[m.env[m.bas[aux, 5]] <= 10.0]
        q[:, 2] = rng.choice(aux, len(q))
        q[250:, 2] = rng.choice(aux[ls[aux] == 1], len(long))
        if name.startswith("int2c2e"):
            q[:, 0], q[:, 1] = rng.choice(aux, len(q)), rng.choice(aux, len(q))
            q[250:, 0] = rng.choice(aux[ls[aux] == 0], len(long))
            q[250:, 1] = rng.choice(aux[ls[aux] == 1], len(long))
        q[:, 3] = 0
    return q


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("omega", [0.0, 0.4, -0.4])
@pytest.mark.parametrize("name", [
    "int2e_sph", "int2e_cart", "int2e_ip1_sph", "int2e_ip1_cart", "int2e_ipip1_sph", "int2e_ip1ip2_cart",
    "int3c2e_sph", "int3c2e_ip1_cart", "int3c2e_ip2_sph", "int2c2e_sph"])
def test_blocks(mc, orc, name, omega, kernel):
    m = _molecule("c4" if "c2e" in name else "c1")
    q = _list(m, name, 21)
    env = m.env.copy()
    env[8] = omega
    with _Route(mc, kernel):
        got, off, nz = mc.batch(name, q, mc.Basis(m.atm, m.bas, env))
    ref, _, nz_r = orc.batch(name, q, orc.Basis(m.atm, m.bas, env))
    size = np.maximum.reduceat(np.abs(ref), off[:-1])
    err = np.maximum.reduceat(np.abs(got - ref), off[:-1])
    bad = np.flatnonzero(err > 1e-12 + 1e-10 * size)
    assert not len(bad), (f"{len(bad)} blocks, the first {q[bad[0]]} (l {m.bas[q[bad[0]], 1]}): "
                          f"{err[bad[0]]:.2e} of {size[bad[0]]:.2e}, largest {err.max():.2e}")
    np.testing.assert_array_equal(nz, nz_r)


@pytest.mark.parametrize("name,ls,nprim,n,omega", [c[:4] + (0.0,) for c in CLASSES]
                         + [("int2e_cart", (4, 2, 3, 0), 2, 1100, -0.4)])
def test_choice_of_kernel(mc, orc, name, ls, nprim, n, omega):
    """One class on the kernel and waves its size, list and primitives choose;
    the exponents are at most 6."""
    m, q = _one_class(ls, nprim, n)
    m.env[8] = omega
    got, off, nz = mc.batch(name, q, mc.Basis(m.atm, m.bas, m.env))
    ref, _, nz_r = orc.batch(name, q, orc.Basis(m.atm, m.bas, m.env))
    size = np.maximum.reduceat(np.abs(ref), off[:-1])
    err = np.maximum.reduceat(np.abs(got - ref), off[:-1])
    assert (err <= 1e-12 + 1e-10 * size).all(), f"{err.max():.2e}"
    np.testing.assert_array_equal(nz, nz_r)


def _dense(orc, m, env):
    """The oracle's (ij|kl) of every shell, as one array."""
    q = unique_quartets(m.nbas)
    out, off, _ = orc.batch("int2e_sph", q, orc.Basis(m.atm, m.bas, env))
    dims = (2 * m.bas[:, 1] + 1) * m.bas[:, 3]
    ao = np.concatenate([[0], np.cumsum(dims)])
    eri = np.zeros((ao[-1],) * 4)
    for n, s in enumerate(q):
        blk = out[off[n]:off[n + 1]].reshape(dims[s], order="F")
        sl = [slice(ao[x], ao[x + 1]) for x in s]
        for t in ((0, 1, 2, 3), (1, 0, 2, 3), (0, 1, 3, 2), (1, 0, 3, 2),
                  (2, 3, 0, 1), (3, 2, 0, 1), (2, 3, 1, 0), (3, 2, 1, 0)):
            eri[tuple(sl[x] for x in t)] = blk.transpose(t)
    return eri


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("omega", [0.0, 0.3])
def test_fused_jk(mc, orc, omega, general):
    """J and K contracted in the kernels, s to f shells, against the dense
    contraction (sums of nao^2 terms of the blocks' accuracy)."""
    from libcint_amd import jk
    m = _molecule("c1", 2)
    m = _general(m) if general else m
    env = m.env.copy()
    env[8] = omega
    eri = _dense(orc, m, env)
    dm = random_density(eri.shape[0], seed=3)
    J, K = np.einsum("ijkl,kl->ij", eri, dm), np.einsum("ijkl,jl->ik", eri, dm)
    for kernel in KERNELS:
        with _Route(mc, kernel):
            vj, vk = jk.get_jk(mc.Basis(m.atm, m.bas, env), dm)
        for got, ref in ((vj, J), (vk, K)):
            np.testing.assert_allclose(got.cpu().numpy(), ref, rtol=0, atol=1e-11 * max(1.0, np.abs(ref).max()),
                                       err_msg=kernel)


def _grad_of_list(mc, B, dm, q):
    import torch
    db = mc.DeviceBasis(B)
    plan = mc.Plan(db, "int2e_ip1_sph", q)
    d = torch.tensor(dm, device="cuda")
    g = torch.zeros((B.natm, 3), dtype=torch.float64, device="cuda")
    plan.execute_grad(d.data_ptr(), dm.shape[0], g.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    db.close()
    return g.cpu().numpy()


@pytest.mark.parametrize("general", [False, True])
def test_gradient_with_f_shells(mc, orc, general):
    """The gradient digest, s to f shells: the reduced list as a program runs
    it (register, matrix and, for (ff|ff), generic kernel) and on the
    runtime-class kernels alone, and the full list, against the oracle's ip1
    blocks contracted on the CPU, to the bound of the other gradient tests."""
    from libcint_amd import jk
    m = _molecule("c1", 3)
    m.bas = m.bas[np.isin(np.arange(m.nbas) % 10, (0, 1, 4, 5, 7, 9))].copy()
    m = _general(m) if general else m
    B = mc.Basis(m.atm, m.bas, m.env)
    dm = random_density(jk.nao_sph(B), seed=11)
    ref = orc.grad_ip1(orc.Basis(m.atm, m.bas, m.env), dm)
    tol = 1e-10 * max(1.0, np.abs(ref).max())
    np.testing.assert_allclose(jk.nuclear_gradient(B, dm, m.natm).cpu().numpy(), ref, rtol=0, atol=tol)
    for kernel in KERNELS:
        with _Route(mc, kernel):
            got = jk.nuclear_gradient(B, dm, m.natm).cpu().numpy()
            full = _grad_of_list(mc, B, dm, jk.gradient_quartets(m.nbas))
        np.testing.assert_allclose(got, ref, rtol=0, atol=tol, err_msg=kernel)
        np.testing.assert_allclose(full, ref, rtol=0, atol=tol, err_msg=kernel)
