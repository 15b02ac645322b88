"""Work-plan tiles: each kind is made by the first call that reads it, and
calls of both kinds may follow each other on one plan in any order."""
import numpy as np
import pytest

from molecules import cluster, random_density
from sqamd import JKEngine

pytestmark = pytest.mark.gpu
CUT = 1e-10


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def test_tiles_made_on_demand():
    mol, bas = cluster(2, 21)
    n = bas.n
    P = random_density(n, 41, 0.05)
    eng = JKEngine(bas.ptr, n)
    b2a = np.arange(n, dtype=np.int32) * 2 // n  # one molecule each
    J, K, _ = (m.copy() for m in eng.build(P, P, CUT, CUT, True))
    nb, nw, _ = eng.plan_tiles()
    assert nb > 0 and nw == 0  # a J/K context makes no wavefront tiles
    eng.class_work()
    nb1, nw1, _ = eng.plan_tiles()
    assert nb1 == nb and nw1 > 0
    G = eng.grad_eri(P, P, b2a, 2, cutoff=16 * CUT)  # the same integral cut-off
    eng.close()

    eng = JKEngine(bas.ptr, n)
    G1 = eng.grad_eri(P, P, b2a, 2, cutoff=16 * CUT)
    nb2, nw2, _ = eng.plan_tiles()
    assert nb2 == 0 and nw2 > 0  # nor a gradient context build tiles
    V = eng.eri_pairs(CUT)
    for cut in (CUT, 1e-6, CUT):  # other plans between, with one kind each
        out = eng.build(P, P, cut, cut, True)
        assert eng.plan_tiles()[0] > 0
    assert _rel(out[0], J) < 1e-13 and _rel(out[1], K) < 1e-13
    assert np.abs(eng.eri_pairs(CUT) - V).max() <= 1e-13
    G2 = eng.grad_eri(P, P, b2a, 2, cutoff=16 * CUT)
    eng.close()
    # forces on whole molecules: sums of terms of the size of J's that cancel
    scale = np.abs(J).max() * np.abs(P).sum()
    assert np.abs(G1 - G).max() <= 1e-13 * scale and np.abs(G2 - G).max() <= 1e-13 * scale


def test_one_plan_for_both_kinds():
    """Build and gradient at one integral cut-off: the second finds the rows of
    the first on the device and adds its own tiles."""
    mol, bas = cluster(3, 22)
    n = bas.n
    P = random_density(n, 42, 0.05)
    b2a = np.arange(n, dtype=np.int32) * 3 // n
    ref = JKEngine(bas.ptr, n)
    G = ref.grad_eri(P, P, b2a, 3, cutoff=16 * CUT)
    ref.close()
    eng = JKEngine(bas.ptr, n)
    out = [m.copy() for m in eng.build(P, P, CUT, CUT, True)]
    st = eng.stats()["quartets"]
    G1 = eng.grad_eri(P, P, b2a, 3, cutoff=16 * CUT)
    again = eng.build(P, P, CUT, CUT, True)
    assert eng.stats()["quartets"] == st
    assert np.abs(G1 - G).max() <= 1e-12 * np.abs(G).max()
    assert all(_rel(a, b) < 1e-13 for a, b in zip(again, out))
    eng.close()
