"""Workgroup tiles of more rows than the workgroup has wavefronts.

Such a tile goes through its rows in several passes, each of which sums the
b-side exchange in accumulators that the pass before left at zero, and its row
list gets long.  (H2O)16/6-31G*: a bra shell meets up to 16 shells of one
kind, so tiles of 9 and more rows exist for every class with a p or d second
shell; J and K against the stored reference values, the UHF build (other
accumulators, half the room) with equal spins against the same ones and with
different spins against tiles of one pass."""
import os

import numpy as np
import pytest

from molecules import random_density
from sqamd import JKEngine, inputs

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
# bra and ket pair class (ss ps pp ds dp dd), wavefronts of the workgroup
SHARED = {"(pp|ps)": (2, 1, 4), "(pp|pp)": (2, 2, 8), "(ds|ps)": (3, 1, 4), "(ds|pp)": (3, 2, 8),
          "(dp|ps)": (4, 1, 8), "(dp|pp)": (4, 2, 8)}


@pytest.fixture(scope="module")
def w16():
    fx = np.load(os.path.join(GOLD, "jk_w16.npz"))
    Z, X = inputs.water_cluster(16, 1601)
    bas = inputs.make_basis(inputs.mol_from_angstrom(Z, X), "631g_star")
    assert bas.n == int(fx["n"])
    eng = JKEngine(bas.ptr, bas.n)
    eng.set_tuning(rows=np.full((6, 6), 64))
    cut = float(fx["cutoff"])
    P = random_density(bas.n, int(fx["seed"]), scale=float(fx["scale"]))
    eng.build(P, P, cut, cut, True)
    deepest = eng.plan_tiles()[2]  # every row of a run in one tile, 64 at most
    yield fx, bas, P, eng, deepest
    eng.close()


@pytest.mark.parametrize("rows", [1, 2, 3, 64])
@pytest.mark.parametrize("restricted", [True, False])
def test_against_reference(w16, rows, restricted):
    fx, bas, P, eng, deepest = w16
    cut = float(fx["cutoff"])
    eng.set_tuning(rows=np.full((6, 6), rows))
    J, KA, KB = eng.build(P, P, cut, cut, restricted)
    longest = eng.plan_tiles()[2]
    for name, (X, Y, waves) in SHARED.items():
        assert longest[X, Y] == min(rows * waves, deepest[X, Y]), name
        if rows == 64 and Y > 0 and X in (2, 4):
            assert longest[X, Y] > waves, name
    r = fx["rows"]
    d = max(np.abs(J[r] - fx["J_rows"]).max(), np.abs(np.diag(J) - fx["Jdiag"]).max())
    for K in (KA,) if restricted else (KA, KB):
        d = max(d, np.abs(K[r] - fx["K_rows"]).max(), np.abs(np.diag(K) - fx["Kdiag"]).max())
    print(f"rows={rows} restricted={restricted}: longest {longest.max()}, max difference {d:.2e}", flush=True)
    assert d < 1e-9


def test_two_spins(w16):
    fx, bas, _, eng, _ = w16
    cut = float(fx["cutoff"])
    PA, PB = random_density(bas.n, 71, 0.05), random_density(bas.n, 72, 0.05)
    out = []
    for rows in (1, 64):
        eng.set_tuning(rows=np.full((6, 6), rows))
        out.append([m.copy() for m in eng.build(PA, PB, cut, cut, False)])
    for a, b in zip(*out):
        # the same integrals in another order: n^2 terms, each below max |b|
        assert np.abs(a - b).max() <= bas.n * np.finfo(float).eps * np.abs(b).max() * 4
