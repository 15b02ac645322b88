"""Results of a batch read a few at a time, in any order, from several threads,
and the cost of reading one."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from molecules import cluster, random_density, water
from sqamd import JKEngine, dptr, inputs, lib
from sqamd.batch import JKBatch

pytestmark = pytest.mark.gpu
CUT = 1e-10


def _small_batch(count, seed):
    inst = inputs.batch_instances(count, seed)
    engines = []
    for x in inst:
        bas = inputs.make_basis(x["mol"], x["basis"])
        engines.append(JKEngine(bas.ptr, bas.n))
    batch = JKBatch(engines, [False] * count)
    batch.set_cutoffs(CUT, CUT)
    return engines, batch


def _set(batch, seed):
    dens = [(random_density(n, seed + 2 * k, 0.05), random_density(n, seed + 2 * k + 1, 0.05))
            for k, n in enumerate(batch.n)]
    for k, d in enumerate(dens):
        batch.set_density(k, *d)
    return dens


def _part(batch, i, which):
    """Only the matrices in `which` of J, K_A, K_B."""
    out = [np.zeros((batch.n[i], batch.n[i])) if k in which else None for k in range(3)]
    rc = lib().sqjk_batch_result(batch._h, i, *[None if m is None else dptr(m) for m in out], 0)
    assert rc == 0
    return out


def test_reads_in_any_order():
    count = 9
    engines, batch = _small_batch(count, 31)
    rng = np.random.default_rng(5)
    for rep in range(4):
        dens = _set(batch, 500 + 50 * rep)
        batch.build(graph=rep > 0)
        ref = [[m.copy() for m in e.build(PA, PB, CUT, CUT, False)] for e, (PA, PB) in zip(engines, dens)]
        order = [list(range(count)), list(range(count))[::-1], [4, 4, 0, 8, 8, 3], rng.permutation(count)][rep]
        for i in order:
            for which in [{0}, {1, 2}, {2}, {0, 1, 2}] if rep % 2 else [{2}, {0, 1, 2}]:
                for k, m in enumerate(_part(batch, i, which)):
                    assert m is None or np.abs(m - ref[i][k]).max() < 1e-12, (rep, i, which, k)
    batch.close()
    for e in engines:
        e.close()


def test_reads_from_threads():
    count = 16
    engines, batch = _small_batch(count, 32)
    dens = [None] * count
    bad = []

    def work(t, phase):
        for i in range(t, count, 4):
            if phase == 0:
                n = batch.n[i]
                dens[i] = random_density(n, 900 + i, 0.05), random_density(n, 950 + i, 0.05)
                batch.set_density(i, *dens[i])
            else:
                ref = engines[i].build(*dens[i], CUT, CUT, False)
                if max(np.abs(a - b).max() for a, b in zip(batch.result(i), ref)) > 1e-12:
                    bad.append(i)

    for phase in range(2):
        if phase:
            batch.build(graph=True)
        threads = [threading.Thread(target=work, args=(t, phase)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    batch.close()
    for e in engines:
        e.close()
    assert bad == []


def test_reading_one_copies_one():
    """Water beside eighty (H2O)16: all matrices are 177 MB, more than 2.5 ms
    over the bus at its nominal 64 GB/s; J of water is 392 bytes."""
    _, wat = water("sto3g")
    _, big = cluster(16, 61)
    engines = [JKEngine(wat.ptr, wat.n), JKEngine(big.ptr, big.n)]
    batch = JKBatch([engines[0]] + 80 * [engines[1]], 81 * [True])
    batch.set_cutoffs(1e-2, 1e-2)
    P = random_density(wat.n, 7)
    batch.set_density(0, P, P)
    lib().sqjk_batch_result.argtypes = [C.c_void_p, C.c_int] + 3 * [C.POINTER(C.c_double)] + [C.c_int]
    ref = engines[0].build(P, P, 1e-2, 1e-2, True)[0]
    times = []
    for rep in range(5):
        batch.build(graph=False)
        t0 = time.perf_counter()
        J = _part(batch, 0, {0})[0]
        times.append(time.perf_counter() - t0)
        assert np.abs(J - ref).max() < 1e-12
    print(f"one J of 7 x 7: {np.median(times) * 1e6:.0f} us", flush=True)
    batch.close()
    for e in engines:
        e.close()
    assert np.median(times) < 1e-3
