"""Launch shapes chosen by the size of a list, against the CPU oracle.

Tolerance: the suite's |gpu - oracle| <= 1e-12 + 1e-10 |oracle| per element
(sums over the same primitives in another order differ by rounding only).
"""
import numpy as np
import pytest

from libcint_amd.synthetic import make_molecule

pytestmark = pytest.mark.gpu


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


def _close(got, ref, what):
    err = np.abs(got - ref)
    bad = err > 1e-12 + 1e-10 * np.abs(ref)
    assert not bad.any(), f"{what}: {int(bad.sum())} elements, max |err| {err.max():.2e}"


def _quartets(nbas, n, seed):
    return np.random.default_rng(seed).integers(0, nbas, (n, 4)).astype(np.int32)


@pytest.mark.parametrize("fill", [0, 1 << 11, 1 << 17, 1 << 30])
@pytest.mark.parametrize("name", ["int2e_sph", "int2e_cart", "int3c2e_sph"])
def test_widened_teams(mc, orc, name, fill):
    """Teams as tuned (0), widened a little and widened to a whole wave give
    the oracle's blocks and flags; contractions of 1 to 10 primitives."""
    m = make_molecule("c4" if name == "int3c2e_sph" else "c1")
    q = _quartets(m.nbas if m.aux_start < 0 else m.aux_start, 700, 5)
    if m.aux_start >= 0:
        q[:, 2] = np.random.default_rng(6).integers(m.aux_start, m.nbas, len(q))
    old = mc.tune(mc.TUNE_FILL_LANES, fill)
    try:
        got, _, nz = mc.batch(name, q, mc.Basis(m.atm, m.bas, m.env))
    finally:
        mc.tune(mc.TUNE_FILL_LANES, old)
    ref, _, nz_r = orc.batch(name, q, orc.Basis(m.atm, m.bas, m.env))
    _close(got, ref, f"{name} fill {fill}")
    np.testing.assert_array_equal(nz, nz_r)


@pytest.mark.parametrize("name,lmax,n", [("int3c2e_ip1_sph", 4, 40000), ("int3c2e_ip2_cart", 4, 34000),
                                         ("int2e_ipip1_sph", 1, 33000), ("int2e_ip1ip2_sph", 3, 300)])
def test_generic_kernel_lists(mc, orc, name, lmax, n):
    """The generic kernel with one task per wave (short lists) and several
    (long buckets), blocks in LDS and (f shells) in global scratch."""
    m = make_molecule("c4" if "3c2e" in name else "c1")
    rng = np.random.default_rng(8)
    ls = m.bas[:, 1]
    orb = np.flatnonzero((ls <= lmax) & (np.arange(m.nbas) < (m.aux_start if m.aux_start >= 0 else m.nbas)))
    if "3c2e" in name:
        # few shells: buckets of tens of thousands of tasks
        orb = np.concatenate([orb[ls[orb] == l][:4] for l in range(4)])
    elif lmax == 1:
        orb = np.concatenate([orb[(ls[orb] == l) & (m.bas[orb, 2] == 1)][:6] for l in range(2)])
    q = rng.choice(orb, (n, 4)).astype(np.int32)
    if "3c2e" in name:
        q[:, 2] = rng.integers(m.aux_start, m.nbas, n)
        q[n // 2:, :2] = orb[:2]
        q[n // 2:, 2] = m.aux_start + rng.integers(0, 12, n - n // 2)
    elif lmax == 3:
        q[:40] = rng.choice(np.flatnonzero(ls == 3), (40, 4))
    B = mc.Basis(m.atm, m.bas, m.env)
    got, off, nz = mc.batch(name, q, B)
    ref, _, nz_r = orc.batch(name, q, orc.Basis(m.atm, m.bas, m.env))
    # the reference transfers weighted sets per primitive; its own rounding
    # on a block is relative to the block's largest intermediate
    for i in range(n):
        s = slice(off[i], off[i + 1])
        scale = max(1.0, np.abs(ref[s]).max(initial=0.0))
        assert np.abs(got[s] - ref[s]).max(initial=0.0) <= 1e-11 * scale + 1e-12, (name, q[i])
    np.testing.assert_array_equal(nz, nz_r)


def _grad_full(mc, B, m, dm):
    """The gradient digest over every (i, j, k >= l)."""
    import torch
    from libcint_amd import jk
    db = mc.DeviceBasis(B)
    plan = mc.Plan(db, "int2e_ip1_sph", jk.gradient_quartets(m.nbas))
    d = torch.tensor(dm, device="cuda")
    g = torch.zeros((m.natm, 3), dtype=torch.float64, device="cuda")
    plan.execute_grad(d.data_ptr(), dm.shape[0], g.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    db.close()
    return g.cpu().numpy()


def _gc_basis(m):
    """m with its first s shell given a second contraction column."""
    bas, env = m.bas.copy(), m.env
    s = int(np.flatnonzero((bas[:, 1] == 0) & (bas[:, 2] > 1))[0])
    n, pc = int(bas[s, 2]), int(bas[s, 6])
    col = env[pc:pc + n]
    bas[s, 3], bas[s, 6] = 2, len(env)
    return bas, np.concatenate([env, col, col[::-1]])


@pytest.mark.parametrize("case", ["atom", "pair", "mol", "general"])
def test_gradient_list(mc, case):
    """Translational invariance: the reduced list's gradient equals the full
    list's (the same sums but for rounding, 1e-10 of the largest), holds no
    derivative on a reference atom, and its plan stores no blocks."""
    from libcint_amd import jk
    from libcint_amd.synthetic import random_density, subset
    m = subset(make_molecule("c3"), {"atom": 1, "pair": 2, "mol": 4, "general": 3}[case])
    bas, env = _gc_basis(m) if case == "general" else (m.bas, m.env)
    B = mc.Basis(m.atm, bas, env)
    dm = random_density(jk.nao_sph(B), seed=4)
    gp = jk.GradientPlan(B, m.natm)
    got = gp.run(dm).cpu().numpy()
    q, refs = gp.db.gradient_list()
    assert gp.nquartets == len(q) == len(refs)
    assert len(q) <= 3 * len(jk.gradient_quartets(m.nbas)) // 4
    atom = bas[:, 0]
    assert (atom[q[:, 0]] != refs).all() and (q[:, 2] >= q[:, 3]).all()
    assert (atom[q] == refs[:, None]).any(axis=1).all()
    for plan in gp.plans:
        with pytest.raises(mc.McintError):
            plan.execute(1 << 12, graph=False)
    gp.close()
    ref = _grad_full(mc, B, m, dm)
    np.testing.assert_allclose(got, ref, rtol=0, atol=1e-10 * max(1.0, np.abs(ref).max()))


@pytest.mark.parametrize("name,omega", [(n, w) for n in (
    "int2e_ipip1_sph", "int2e_ipip1_cart", "int2e_ip1ip2_sph", "int2e_ip1ip2_cart", "int3c2e_ip1_sph",
    "int3c2e_ip2_cart", "int2c2e_sph") for w in (0.0, 0.4, -0.4)] + [("int2e_cart", -0.4)])
def test_matrix_kernel(mc, orc, name, omega):
    """Plans on the matrix kernel: every order of s, p, d (and one f, one g)
    shells, one and four waves per task (buckets below and above 1024 tasks),
    1 to 4096 primitive quartets, all operators."""
    m = make_molecule("c4" if "c2e" in name else "c1")
    rng = np.random.default_rng(12)
    ls, three = m.bas[:, 1], "c2e" in name
    ns = m.aux_start if m.aux_start >= 0 else m.nbas
    orb = np.arange(ns)
    few = [orb[ls[:ns] == l][:5] for l in range(4)]
    deep = [orb[(ls[:ns] == l) & (m.bas[:ns, 2] > 1)][:1] for l in range(2)]
    pool = np.concatenate(few[:3] + deep)
    q = rng.choice(pool, (260, 4)).astype(np.int32)
    q[:4, 0] = few[3][0]
    q[4:8, 2] = few[3][0]
    short = rng.choice(np.concatenate([orb[(ls[:ns] == l) & (m.bas[:ns, 2] == 1)][:4] for l in range(2)]), (1, 4))
    q = np.concatenate([q, np.repeat(short, 1100, axis=0)]).astype(np.int32)
    if three:
        aux = np.arange(m.aux_start, m.nbas)
        q[:, 2] = rng.choice(aux, len(q))
        q[260:, 2] = aux[ls[aux] == 0][0]
        if name.startswith("int2c2e"):
            q[:, 0], q[:, 1] = rng.choice(aux, len(q)), rng.choice(aux, len(q))
        q[:, 3] = 0
    env = m.env.copy()
    env[8] = omega
    got, off, nz = mc.batch(name, q, mc.Basis(m.atm, m.bas, env))
    ref, _, nz_r = orc.batch(name, q, orc.Basis(m.atm, m.bas, env))
    # as for the generic kernel: relative to the block's largest element
    for i in range(len(q)):
        s = slice(off[i], off[i + 1])
        scale = max(1.0, np.abs(ref[s]).max(initial=0.0))
        assert np.abs(got[s] - ref[s]).max(initial=0.0) <= 1e-11 * scale + 1e-12, (name, omega, q[i])
    np.testing.assert_array_equal(nz, nz_r)


@pytest.mark.parametrize("name", ["int2e_ip1_sph", "int2e_ip1_cart", "int2e_ip2_sph"])
@pytest.mark.parametrize("omega", [0.0, 0.3])
def test_derivative_wave_kernel(mc, name, omega):
    """Derivative classes on the wave kernel (every class that has one, one to
    1296 primitive quartets, odd counts per wave) against the chunk kernels:
    the same sums in another order."""
    m = make_molecule("c3")
    ls, env = m.bas[:, 1], m.env.copy()
    env[8] = omega
    rng = np.random.default_rng(3)
    pool = np.concatenate([np.flatnonzero(ls == l)[:6] for l in range(3)])
    q = rng.choice(pool, (1501, 4)).astype(np.int32)
    out = []
    old = mc.tune(mc.TUNE_WAVE_KERNELS, 0)
    try:
        for mode in (0, 2):
            mc.tune(mc.TUNE_WAVE_KERNELS, mode)
            out.append(mc.batch(name, q, mc.Basis(m.atm, m.bas, env)))
    finally:
        mc.tune(mc.TUNE_WAVE_KERNELS, old)
    (a, _, nza), (b, _, nzb) = out
    scale = max(1.0, np.abs(a).max())
    assert np.abs(a - b).max() <= 1e-12 * scale
    np.testing.assert_array_equal(nza, nzb)


def test_gradient_wave_kernel(mc):
    """The gradient through wave and chunk kernels, waves taking many quartets."""
    from libcint_amd import jk
    from libcint_amd.synthetic import random_density, subset
    m = subset(make_molecule("c3"), 4)
    B = mc.Basis(m.atm, m.bas, m.env)
    dm = random_density(m.nao_sph(), seed=9)
    out = []
    old = mc.tune(mc.TUNE_WAVE_KERNELS, 0)
    try:
        for mode in (0, 1, 2):
            mc.tune(mc.TUNE_WAVE_KERNELS, mode)
            out.append(jk.nuclear_gradient(B, dm, m.natm).cpu().numpy())
    finally:
        mc.tune(mc.TUNE_WAVE_KERNELS, old)
    for g in out[1:]:
        np.testing.assert_allclose(g, out[0], rtol=0, atol=1e-11 * max(1.0, np.abs(out[0]).max()))


def test_large_host_batches(mc):
    """Lists and outputs beyond the staging buffers' size: a host batch equals
    the same plan's device buffer, from several threads at once as alone."""
    import threading

    import torch
    from libcint_amd.synthetic import subset, unique_quartets
    m = subset(make_molecule("c3"), 7)
    B = mc.Basis(m.atm, m.bas, m.env)
    q = unique_quartets(m.nbas)
    assert q.nbytes > 4 << 20
    db = mc.DeviceBasis(B)
    plan = mc.Plan(db, "int2e_sph", q)
    dev = torch.full((plan.out_size,), 7.0, dtype=torch.float64, device="cuda")
    plan.execute(dev.data_ptr(), graph=False)
    ref = dev.cpu().numpy()
    plan.close()
    db.close()
    assert ref.nbytes > 3 * (2 << 20) + 8
    got = [None] * 4

    def work(i):
        got[i] = mc.batch("int2e_sph", q[:len(q) - i], B)[0]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        np.testing.assert_allclose(g, ref[:len(g)], rtol=0, atol=1e-13)
