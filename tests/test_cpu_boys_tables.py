"""The tabulated Boys functions (eri_math.h) against the reference's procedure
(Taylor sum of F_Q about Tk, downward recursion; asymptotic above T = 12,
auxilary.f90:130-215) in 80-bit arithmetic: at the middle and both ends of the
table's intervals, and on both sides of the procedure's own limits.

Tolerance (relative): below T = 12 the telescoped series is within 1.2e-15 of
the procedure, e^-T's series within 1e-15, and x and the M <= 4 downward steps
add an ulp or two each; above, F_4 is the ninth power of 1/sqrt(T) (within 1.5
ulp) in eight more roundings.  Either stays below 4e-15."""
import ctypes
import os

import numpy as np
import pytest

from myqc_amd.basis import read_ftab

_dp = ctypes.POINTER(ctypes.c_double)
HC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hostcheck", "libhostcheck.so")
L = np.longdouble
PI = L(np.float32(3.1415926535897931))


def _procedure(Q, T, F):
    """F_0 .. F_4 (zero above Q)"""
    T, out = L(T), np.zeros(5, L)
    if T < 12:
        k = int(np.floor(10 * T + L(0.5)))
        x = L(k) / 10 - T
        f = sum(L(F[Q + i, k]) * x ** i / L(float(np.prod(np.arange(1.0, i + 1)))) for i in range(7))
        for j in range(Q, -1, -1):
            if j < Q:
                f = (2 * T * f + np.exp(-T)) / (2 * j + 1)
            if j <= 4:
                out[j] = f
        return out
    near = T < 2 * Q + 36
    g = L(0)
    if near:
        c = ([0.4999489092, -0.2473631686, 0.321180909, -0.3811559346] if T < 15 else
             [0.4998436875, -0.24249438, 0.24642845] if T < 18 else [0.499093162, -0.2152832] if T < 24 else [0.490])
        g = sum(L(v) * T ** -i for i, v in enumerate(c))
    e = np.exp(-T) if near else L(0)
    out[0] = np.sqrt(PI) / 2 / np.sqrt(T) - e * g / T
    for j in range(1, 5):
        out[j] = ((2 * j - 1) * out[j - 1] - e) / (2 * T)
    return out


@pytest.mark.parametrize("Q", [0, 3, 6, 9, 12])
def test_boys_tables(Q):
    if not os.path.exists(HC):
        pytest.skip("host check harness not built (run __graft_entry__.build())")
    hc = ctypes.CDLL(HC)
    ftab = np.ascontiguousarray(read_ftab(), dtype=np.float64)
    F = ftab.reshape(-1, 121)
    mid = np.arange(120) / 10.0
    T = np.concatenate([mid, mid + 0.049999, mid + 0.050001, [11.96, 12 - 1e-9, 12, 14.999, 15, 18, 24, 35.99, 36],
                        [2 * Q + 36 - 1e-9, 2 * Q + 36, 59.97, 61, 1e4]])
    got = np.zeros(5)
    for M in range(5):
        for t in T:
            assert hc.hc_boys(M, Q, ctypes.c_double(float(t)), ftab.ctypes.data_as(_dp), got.ctypes.data_as(_dp)) == 0
            ref = _procedure(Q, float(t), F)
            for j in range(min(M, Q) + 1):
                assert abs(L(got[j]) - ref[j]) <= 4e-15 * abs(ref[j]), (M, j, t)
