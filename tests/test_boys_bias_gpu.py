"""FP32 Boys function: its errors must not lean one way.

A J/K element sums up to millions of FP32 integrals.  Independent roundings
average out, a common bias does not.  F_L by Taylor expansion about the
nearest grid point takes a handful of roundings of 6e-8 (half a unit in the
last place), so over 40,000 random arguments the mean relative error of an
unbiased evaluation is below 6e-8 * sqrt(10) / 200 = 1e-9 from rounding, plus
the rounding of the table's own entries, which a quarter of 6e-8 leaves room
for (each argument interval of 0.1 has its own)."""
import ctypes as C

import numpy as np
import pytest
from scipy.special import gamma, gammainc

from sqamd import dptr, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", list(range(10)))
def test_fp32_boys_unbiased(L):
    T = np.random.default_rng(40 + L).uniform(0.1, 30.0, 40000).astype(np.float32).astype(np.float64)
    ref = gammainc(L + 0.5, T) * gamma(L + 0.5) / (2 * T ** (L + 0.5))
    F = np.zeros((len(T), L + 1))
    lib().sqjk_boys.argtypes = [C.c_int, C.c_int, C.POINTER(C.c_double), C.c_int, C.c_int, C.POINTER(C.c_double)]
    assert lib().sqjk_boys(L, len(T), dptr(T), 1, 0, dptr(F)) == 0, lib().sqjk_errmsg()
    mean = ((F[:, L] - ref) / ref).mean()
    print(f"L={L}: mean relative error {mean:.2e}", flush=True)
    assert abs(mean) < 2.0 ** -26


@pytest.mark.parametrize("L", list(range(1, 10)))
def test_fp32_boys_recursion_unbiased(L):
    T = np.random.default_rng(60 + L).uniform(0.1, 30.0, 40000).astype(np.float32).astype(np.float64)
    F = np.zeros((len(T), L + 1))
    lib().sqjk_boys.argtypes = [C.c_int, C.c_int, C.POINTER(C.c_double), C.c_int, C.c_int, C.POINTER(C.c_double)]
    assert lib().sqjk_boys(L, len(T), dptr(T), 1, 0, dptr(F)) == 0, lib().sqjk_errmsg()
    mean = []
    for m in range(L):
        ref = gammainc(m + 0.5, T) * gamma(m + 0.5) / (2 * T ** (m + 0.5))
        mean.append(((F[:, m] - ref) / ref).mean())
    print(f"L={L}: mean relative errors " + " ".join(f"{x:.1e}" for x in mean), flush=True)
    assert max(abs(x) for x in mean) < 2.0 ** -26
