"""With MCINT_TUNE_FILL_LANES 0 a tuple's block does not depend on its list:
the same bits alone, among a few others and in a long list."""
import numpy as np
import pytest

from libcint_amd.synthetic import make_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["int2e_sph", "int2e_cart", "int2e_ip1_sph", "int2e_ipip1_sph", "int2e_ip1ip2_sph",
                                  "int3c2e_sph", "int3c2e_ip1_sph", "int3c2e_ip2_cart", "int2c2e_sph"])
@pytest.mark.parametrize("omega", [0.0, -0.3])
def test_bits_of_a_block(name, omega):
    import libcint_amd as mc
    m = make_molecule("c4" if "c2e" in name else "c3")
    rng = np.random.default_rng(4)
    ns = m.aux_start if m.aux_start >= 0 else m.nbas
    shells = rng.choice(ns, 12, replace=False)
    q = rng.choice(shells, (6000, 4)).astype(np.int32)
    if m.aux_start >= 0:
        aux = rng.choice(np.arange(m.aux_start, m.nbas), 12, replace=False)
        q[:, 2] = rng.choice(aux, len(q))
        if name.startswith("int2c2e"):
            q[:, 0], q[:, 1] = rng.choice(aux, len(q)), rng.choice(aux, len(q))
    env = m.env.copy()
    env[8] = omega
    B = mc.Basis(m.atm, m.bas, env)
    old = mc.tune(mc.TUNE_FILL_LANES, 0)
    try:
        whole, off, _ = mc.batch(name, q, B)
        for part in (np.arange(40, 41), np.arange(100, 163), np.arange(1, 6000, 7)):
            got, o, _ = mc.batch(name, q[part], B)
            for n, t in enumerate(part):
                np.testing.assert_array_equal(got[o[n]:o[n + 1]], whole[off[t]:off[t + 1]], err_msg=str(q[t]))
    finally:
        mc.tune(mc.TUNE_FILL_LANES, old)


def _class_list(m, ls, n):
    rng = np.random.default_rng(6)
    one = [np.flatnonzero((m.bas[:, 1] == l) & (m.bas[:, 2] == 1))[:6] for l in ls]
    return np.stack([rng.choice(x, n) for x in one], axis=1).astype(np.int32)


@pytest.mark.parametrize("ls,wave", [((1, 2, 1, 1), False), ((2, 2, 1, 1), False), ((1, 2, 2, 1), False),
                                     ((2, 1, 2, 1), True)])
def test_derivative_class_by_its_list(ls, wave):
    """Long lists of the derivative classes with few columns run the chunk
    kernels (8192 tuples and more), shorter ones the wave kernel, each with its
    own bits; with 0 lanes to fill the list makes no difference."""
    import libcint_amd as mc
    m = make_molecule("c3")
    B = mc.Basis(m.atm, m.bas, m.env)
    q = _class_list(m, ls, 8192)

    def run(n, **keys):
        old = {k: mc.tune(getattr(mc, k), v) for k, v in keys.items()}
        try:
            return mc.batch("int2e_ip1_sph", q[:n], B)[0]
        finally:
            for k, v in old.items():
                mc.tune(getattr(mc, k), v)

    tuned = {"TUNE_FILL_LANES": 1 << 17}
    chunk, waves = run(8192, TUNE_WAVE_KERNELS=0, **tuned), run(8192, TUNE_WAVE_KERNELS=2, **tuned)
    np.testing.assert_array_equal(run(8192, **tuned), waves if wave else chunk)
    short = run(8191, **tuned)
    np.testing.assert_array_equal(short, waves[:len(short)])
    fixed = run(8192, TUNE_FILL_LANES=0)
    np.testing.assert_array_equal(run(50, TUNE_FILL_LANES=0), fixed[:len(fixed) // 8192 * 50])
    np.testing.assert_allclose(chunk, waves, rtol=0, atol=1e-12 * max(1.0, np.abs(chunk).max()))
