"""Component scales and permutation weights of FP32 quartets enter in FP64.

Scaling the later components of a shell by s_p leaves the shell's radial part,
and with it every FP32 quantity, as it was: an integral picks up s_p s_q s_r
s_t.  With the density divided by s_r s_t, J and K of the scaled basis must be
s_p s_q times those of the plain one to FP64 rounding.  A scale that took part
in the FP32 products would leave its rounding, 6e-8 of every integral."""
import numpy as np
import pytest

from molecules import cluster, random_density
from sqamd import JKEngine
from sqamd.abi import Basis, basis_from_ptr
from sqamd.batch import JKBatch

pytestmark = pytest.mark.gpu
ALL_FP32 = 1e6  # Schwarz products are far below it


def _scaled(bas):
    """The basis with every component but a shell's first scaled, and the scales."""
    s = np.ones(bas.n)
    funcs = []
    for i, (l, m, n, c, ex, co, no) in enumerate(basis_from_ptr(bas.ptr, bas.n)):
        if l + m + n > 0 and l != l + m + n:
            s[i] = 0.7 + 0.045 * (i % 13)
        funcs.append((l, m, n, c, ex, co, no * s[i]))
    return Basis(funcs), s


def _check(plain, scaled, s, sch, densities):
    """Every element sums at most n^2 integrals of at most max(sch)^2, in FP64."""
    n = len(s)
    bound = n * n * np.finfo(float).eps * sch.max() ** 2 * 2 * max(np.abs(D).sum() for D in densities)
    d = max(np.abs(b / np.outer(s, s) - a).max() for a, b in zip(plain, scaled))
    print(f"n={n}: max difference {d:.2e}, bound {bound:.2e}", flush=True)
    assert d <= bound


@pytest.mark.parametrize("restricted", [True, False])
@pytest.mark.parametrize("thr", [1e-4, ALL_FP32])
def test_scaled_components(thr, restricted):
    mol, bas = cluster(2, 11, "631g_star")
    n = bas.n
    PA = random_density(n, 31)
    PB = PA if restricted else random_density(n, 32)
    sbas, s = _scaled(bas)
    eng = JKEngine(bas.ptr, n)
    sch = eng.schwarz()
    eng.close()
    out = []
    for b, t in ((bas, np.ones(n)), (sbas, s)):
        eng = JKEngine(b.ptr, n, schwarz=sch)
        eng.set_mixed(thr)
        D = np.outer(t, t)
        out.append([m.copy() for m in eng.build(PA / D, PB / D, 0.0, 0.0, restricted)])
        assert eng.stats()["quartets_fp32"] > 0
        eng.close()
    _check(out[0], out[1], s, sch, (PA + PB,))


def test_scaled_components_batch():
    mol, bas = cluster(2, 12, "631g_star")
    n = bas.n
    PA, PB = random_density(n, 33), random_density(n, 34)
    sbas, s = _scaled(bas)
    eng = JKEngine(bas.ptr, n)
    sch = eng.schwarz()
    eng.close()
    engines = [JKEngine(b.ptr, n, schwarz=sch) for b in (bas, sbas)]
    batch = JKBatch(engines, [False, False])
    batch.set_cutoffs(0.0, 0.0)
    batch.set_mixed(ALL_FP32)
    D = np.outer(s, s)
    batch.set_density(0, PA, PB)
    batch.set_density(1, PA / D, PB / D)
    batch.build(graph=False)
    out = [[m.copy() for m in batch.result(k)] for k in range(2)]
    batch.close()
    for e in engines:
        e.close()
    _check(out[0], out[1], s, sch, (PA + PB,))
