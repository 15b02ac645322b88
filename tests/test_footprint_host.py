"""sqjk_footprint_bytes, by which served requests are admitted, covers what a
context allocates, counted here from the basis, and little more (no device
needed)."""
import ctypes as C

import pytest

from molecules import cluster, water
from sqamd import lib
from sqamd.workmodel import cart, ncart

CLASS = [(0, 0), (1, 0), (1, 1), (2, 0), (2, 1), (2, 2)]


def _table_stride(la, lb):
    """Bra products of a primitive pair: (nx+1)(ny+1)(nz+1) for each pair of
    components, padded to 16; none for ss."""
    terms = 0
    for a in range(ncart(la)):
        for b in range(ncart(lb)):
            k = 1
            for x, y in zip(cart(la, a), cart(lb, b)):
                k *= x + y + 1
            terms += k
    return 0 if la + lb == 0 else (terms + 15) // 16 * 16


def _shells(bas):
    """(l, primitives) of every pure shell: first components only."""
    out = []
    for i in range(bas.n):
        g = bas.ptr[i]
        if g.l == g.l + g.m + g.n:
            out.append((g.l, g.nContract))
    return out


@pytest.mark.parametrize("uhf", [False, True])
@pytest.mark.parametrize("make", [lambda: water("sto3g"), lambda: cluster(2, 3, "631g"), lambda: cluster(4, 5, "631g"),
                                  lambda: cluster(8, 7, "631g")])
def test_covers_every_buffer(make, uhf):
    _, bas = make()
    n, sh = bas.n, _shells(bas)
    npair, nprim = [0] * 6, [0] * 6
    for i, (li, pi) in enumerate(sh):
        for lj, pj in sh[:i + 1]:
            X = CLASS.index((max(li, lj), min(li, lj)))
            npair[X] += 1
            nprim[X] += pi * pj
    need = 12 * n * n * 8 + len(sh) * 48 + n * 8  # matrices, shells, component scales
    need += 651 * 29 * 8                          # Boys table
    for X, (la, lb) in enumerate(CLASS):
        need += npair[X] * (40 + 8 * ncart(la) * ncart(lb))                        # pairs, J by pair
        need += npair[X] * n * (ncart(la) + ncart(lb)) * 8 * (2 if uhf else 1)     # exchange staging
        need += nprim[X] * (64 + _table_stride(la, lb) * (8 + 4))                  # primitives, FP64 and FP32 bra tables
    L = lib()
    L.sqjk_footprint_bytes.restype = C.c_longlong
    got = L.sqjk_footprint_bytes(n, bas.ptr, int(uhf), 0)
    print(f"n={n} uhf={uhf}: counted {need}, estimate {got} with an eighth for the work plan")
    # screening maxima, work buffers of a page each
    assert need <= got * 8 / 9 <= 1.02 * need + 16384
