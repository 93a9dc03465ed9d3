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
