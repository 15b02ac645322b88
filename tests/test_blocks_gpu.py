"""The block cache on the device: what MP2 keeps for its next call goes with
sqjk_release_cached and with the context, and changes no result."""
import ctypes as C

import numpy as np
import pytest

from molecules import cluster, random_density
from sqamd import JKEngine, lib, release_cached

pytestmark = pytest.mark.gpu


def _orbitals(n, seed):
    """Orthonormal columns and orbital energies with a gap above the first third."""
    q, _ = np.linalg.qr(random_density(n, seed))
    return np.sort(np.concatenate([-1.0 - np.arange(n // 3) / n, 0.5 + np.arange(n - n // 3) / n])), np.ascontiguousarray(q.T)


def test_release_between_calls():
    mol, bas = cluster(4, 17, "631g_star")  # n = 76: a pair matrix of 69 MB
    n = bas.n
    e, Cm = _orbitals(n, 3)
    eng = JKEngine(bas.ptr, n)
    release_cached()
    first = eng.mp2_rhf(n // 3, 0, e, Cm)["e2"]
    V = eng.eri_pairs()
    assert release_cached() >= V.nbytes  # the pair matrix was kept
    assert release_cached() == 0
    again = eng.mp2_rhf(n // 3, 0, e, Cm)["e2"]
    assert abs(again - first) <= 1e-12 * abs(first)
    assert np.abs(eng.eri_pairs() - V).max() <= 1e-13  # split tiles add in any order
    eng.close()


def test_large_blocks_go_with_the_context():
    mol, bas = cluster(10, 18, "631g_star")  # n = 190: a pair matrix of 2.6 GB
    n = bas.n
    e, Cm = _orbitals(n, 4)
    m = n * (n + 1) // 2
    other = JKEngine(bas.ptr, n)
    eng = JKEngine(bas.ptr, n)
    release_cached()
    eng.mp2_rhf(n // 3, 0, e, Cm, 1e-10)
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def available():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    before = available()
    eng.close()
    print(f"{(available() - before) >> 20} MiB given back, pair matrix {m * m * 8 >> 20} MiB", flush=True)
    assert available() - before >= m * m * 8  # while another context is alive
    other.close()
    release_cached()
