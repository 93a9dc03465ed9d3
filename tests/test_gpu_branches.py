"""Launches that are not captured on one to eight side streams: the J/K and the
gradient sum the same terms (rounding only), a host batch writes the same bits."""
import numpy as np
import pytest

from libcint_amd.synthetic import make_molecule, random_density, subset, unique_quartets

pytestmark = pytest.mark.gpu


def test_side_streams():
    import libcint_amd as mc
    from libcint_amd import jk
    m = subset(make_molecule("c3"), 4)
    B = mc.Basis(m.atm, m.bas, m.env)
    q = unique_quartets(m.nbas)
    dm = random_density(m.nao_sph(), seed=2)
    got = {}
    for n in (1, 2, 3, 4, 6, 8):
        old = mc.tune(mc.TUNE_GRAPH_BRANCHES, n)
        try:
            vj, vk = jk.get_jk(B, dm)
            got[n] = [vj.cpu().numpy(), vk.cpu().numpy(), jk.nuclear_gradient(B, dm, m.natm).cpu().numpy(),
                      mc.batch("int2e_sph", q, B)[0]]
        finally:
            mc.tune(mc.TUNE_GRAPH_BRANCHES, old)
    for n, g in got.items():
        for a, b in zip(g[:3], got[1][:3]):
            np.testing.assert_allclose(a, b, rtol=0, atol=1e-12 * max(1.0, np.abs(b).max()), err_msg=str(n))
        np.testing.assert_array_equal(g[3], got[1][3], err_msg=str(n))
