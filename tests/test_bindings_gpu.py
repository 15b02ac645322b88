"""The library's functions are shared by all Python code of a process: a
program that declares sqjk_one_electron or nuclei_coulomb with the structure
of the header leaves DeviceSCF's own calls working, in either order."""
import ctypes as C

import numpy as np
import pytest

from molecules import g2
from sqamd import GTOBasis, Molecule, lib
from sqamd.scf import DeviceSCF, one_electron

pytestmark = pytest.mark.gpu
PD = C.POINTER(C.c_double)


@pytest.mark.parametrize("arg", [C.POINTER(Molecule), C.c_void_p])
def test_declared_by_the_caller_too(arg):
    mol, bas = g2("h2o_q0m1", "sto3g")
    H0, S0 = one_electron(bas, mol)
    L = lib()
    names = ("sqjk_one_electron", "nuclei_coulomb")
    before = [getattr(L, f).argtypes for f in names]
    L.sqjk_one_electron.argtypes = [C.c_int, C.POINTER(GTOBasis), arg, C.c_int, PD, PD, PD]
    L.nuclei_coulomb.argtypes = [arg]
    try:
        scf = DeviceSCF()
        H, S = scf.set_system(bas, mol)
        scf.diag_guess(S, 5, 5)
        r = scf.run(5, 5)
        scf.close()
    finally:
        for f, a in zip(names, before):
            getattr(L, f).argtypes = a
    assert np.array_equal(H, H0) and np.array_equal(S, S0)
    assert r["converged"]
