"""Host batches' copies back to pageable memory.

The same kernels write the same bits for the same list, so blocks and flags
are compared for equality.
"""
import ctypes
import threading

import numpy as np
import pytest

from libcint_amd.synthetic import make_molecule, subset, unique_quartets

pytestmark = pytest.mark.gpu

PER_THREAD_STREAM = 2  # HIP's hipStreamPerThread


@pytest.fixture(scope="module")
def mc():
    import libcint_amd
    libcint_amd.lib()
    return libcint_amd


@pytest.fixture(scope="module")
def case(mc):
    """A list whose blocks and flags take several staging buffers each."""
    m = subset(make_molecule("c3"), 7)
    B = mc.Basis(m.atm, m.bas, m.env)
    q = np.tile(unique_quartets(m.nbas), (3, 1))
    out, _, nz = mc.batch("int2e_sph", q, B)
    assert out.nbytes > 4 * (2 << 20) and nz.nbytes > 2 << 20
    return B, q, out, nz


def _batch(mc, B, q, size, stream):
    out, nz = np.full(size, 7.0), np.full(len(q), 9, np.int32)
    ip = ctypes.POINTER(ctypes.c_int)
    dp = ctypes.POINTER(ctypes.c_double)
    rc = mc.lib().int2e_sph_batch(out.ctypes.data_as(dp), None, q.ctypes.data_as(ip), len(q),
                                  B.atm.ctypes.data_as(ip), B.natm, B.bas.ctypes.data_as(ip), B.nbas,
                                  B.env.ctypes.data_as(dp), None, nz.ctypes.data_as(ip), stream)
    assert rc == 0
    return out, nz


def _same(got, case):
    np.testing.assert_array_equal(got[0], case[2])
    np.testing.assert_array_equal(got[1], case[3])


@pytest.mark.parametrize("callers", [1, 3])
def test_batch_on_the_per_thread_stream(mc, case, callers):
    """The per-thread stream is another one in each of the copying threads."""
    B, q, out, _ = case
    got = [None] * callers

    def work(i):
        got[i] = _batch(mc, B, q, out.size, PER_THREAD_STREAM)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(callers)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        _same(g, case)


@pytest.mark.parametrize("limit", [0, 1, 3, 16])
def test_batch_without_staging_buffers(mc, case, limit):
    """Threads that get no pinned buffer leave their part to the others, and a
    transfer that gets none goes without; no more exist than the bound."""
    B, q, out, _ = case
    L = mc.lib()
    set_limit, live = L._ZN5mcint11stage_limitEi, L._ZN5mcint11stages_liveEv
    old = set_limit(limit)
    try:
        assert live() == 0
        got = [None] * 3

        def work(i):
            got[i] = _batch(mc, B, q, out.size, None)

        threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert live() <= limit
    finally:
        set_limit(old)
    for g in got:
        _same(g, case)
