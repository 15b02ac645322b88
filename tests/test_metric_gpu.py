"""The metric X = U^-1 of an overlap matrix S = U^T U (sq_linalg.hip): block
edges, matrices without a factor, and solves side by side."""
import ctypes as C
import threading

import numpy as np
import pytest

from molecules import cluster, g2
from sqamd import dptr, lib
from sqamd.scf import DeviceSCF

pytestmark = pytest.mark.gpu
PD = C.POINTER(C.c_double)
EPS = np.finfo(float).eps


def _eigen(F, S):
    L, n = lib(), len(S)
    L.sqla_gen_eigen.argtypes = [C.c_int, PD, PD, PD, PD]
    e, Cm = np.zeros(n), np.zeros((n, n))
    rc = L.sqla_gen_eigen(n, dptr(np.ascontiguousarray(F)), dptr(np.ascontiguousarray(S)), dptr(e), dptr(Cm))
    return rc, e, Cm


def _spd(n, seed, cond):
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    S = (q * np.logspace(0, -np.log10(cond), n)) @ q.T
    return (S + S.T) / 2


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 128, 129, 191, 192, 193, 300])
@pytest.mark.parametrize("cond", [1e1, 1e6])
def test_block_edges(n, cond):
    """F C = S C e against numpy through the Cholesky factor.  Orthonormality
    in S and the eigenvalues lose n eps cond(S) at most."""
    S = _spd(n, n, cond if n > 1 else 1.0)
    A = np.random.default_rng(1000 + n).standard_normal((n, n))
    F = A + A.T
    rc, e, Cm = _eigen(F, S)
    assert rc == 0
    Li = np.linalg.inv(np.linalg.cholesky(S))
    ref = np.linalg.eigvalsh(Li @ F @ Li.T)
    bound = 8 * n * EPS * cond
    orth, de = np.abs(Cm @ S @ Cm.T - np.eye(n)).max(), np.abs(e - ref).max() / np.abs(ref).max()
    print(f"n={n} cond={cond:g}: C S C^T - 1 {orth:.1e}, eigenvalues {de:.1e}, bound {bound:.1e}", flush=True)
    assert orth < bound and de < bound


@pytest.mark.parametrize("n,at", [(1, 1), (50, 1), (50, 50), (100, 64), (100, 65), (200, 128), (200, 200)])
def test_no_factor_is_refused(n, at):
    """The minor `at` is the first that is not positive definite."""
    S = _spd(n, 7 * n, 10.0 if n > 1 else 1.0)
    k = at - 1
    S[k, k] = S[k, :k] @ np.linalg.solve(S[:k, :k], S[:k, k]) - 0.1 if k else -0.1
    assert _eigen(np.eye(n), S)[0] != 0
    S[0, 0] = np.nan
    assert _eigen(np.eye(n), S)[0] != 0
    assert _eigen(np.eye(n), _spd(n, 8 * n, 10.0 if n > 1 else 1.0))[0] == 0  # the next one is not touched by it


def test_solves_side_by_side():
    """Four contexts, each moving between molecules: every solve's orbitals are
    orthonormal in the true overlap and its energy is that of the same solve
    alone (two iterations; the overlap matrices have condition numbers below
    1e4, the energies a few thousand atomic-summation roundings)."""
    mols = [cluster(4, 31, "631g"), cluster(8, 32, "631g"), cluster(12, 33, "631g"), g2("c2h4_q0m1", "631g"),
            cluster(15, 34, "631g")]

    def solve(scf, mol, bas):
        ne = mol.n_electrons // 2
        _, S = scf.set_system(bas, mol)
        scf.diag_guess(S, ne, ne)
        E = scf.run(ne, ne, conv=1e-3, max_iter=2)["energy"]
        return E, np.abs((Cm := scf.orbitals()[0]) @ S @ Cm.T - np.eye(bas.n)).max()

    one = DeviceSCF()
    ref = [solve(one, *m)[0] for m in mols]
    one.close()
    bad, worst = [], [0.0] * 4

    def work(t):
        rng, scf = np.random.default_rng(t), DeviceSCF()
        for it in range(150):
            i = int(rng.integers(len(mols)))
            try:
                E, orth = solve(scf, *mols[i])
            except RuntimeError as ex:
                bad.append((t, it, i, str(ex)))
                scf = DeviceSCF()
                continue
            worst[t] = max(worst[t], orth)
            if orth > 1e-9 or abs(E - ref[i]) > 1e-8:
                bad.append((t, it, i, orth, E - ref[i]))
        scf.close()

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print("600 solves, worst C S C^T - 1", max(worst), "bad", bad[:5], flush=True)
    assert not bad
