"""Work-plan tuning tables: what sqjk_get_tuning returns can be set again."""
import ctypes as C

import numpy as np
import pytest

from molecules import cluster, random_density
from sqamd import JKEngine
from sqamd.batch import _bind

pytestmark = pytest.mark.gpu
CUT = 1e-10


def _get(eng):
    t = [np.zeros(36, dtype=np.int32) for _ in range(3)]
    assert _bind().sqjk_get_tuning(eng._h, *[a.ctypes.data_as(C.POINTER(C.c_int)) for a in t]) == 0
    return [a.reshape(6, 6) for a in t]


def test_set_what_get_returned():
    """Neither the build's tiles nor those of the gradient and the integral
    store change, at once and after other tables in between."""
    mol, bas = cluster(4, 23)
    n = bas.n
    P = random_density(n, 43, 0.05)
    b2a = np.zeros(n, dtype=np.int32)
    eng = JKEngine(bas.ptr, n)

    def tiles():
        eng.build(P, P, CUT, CUT, True)
        eng.class_work()  # wavefront tiles of the same plan
        nb, nw, longest = eng.plan_tiles()
        eng.grad_eri(P, P, b2a, 1)
        return nb, nw, longest.tolist(), eng.plan_tiles()[1]

    first, table = tiles(), _get(eng)
    eng.set_tuning(*table)
    assert tiles() == first
    eng.set_tuning(rows=np.full((6, 6), 5))
    assert tiles() != first
    eng.set_tuning(*table)
    assert tiles() == first
    eng.set_tuning(rows=np.full((6, 6), 1))
    ones = tiles()
    eng.set_tuning(*_get(eng))
    assert tiles() == ones
    eng.set_tuning()  # defaults
    assert tiles() == first and all((a == b).all() for a, b in zip(_get(eng), table))
    eng.close()
