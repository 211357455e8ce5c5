"""RHF of a small system whose core Hamiltonian holds a not-a-number: the call
reports that it did not converge, and its energy and orbital energies are not
numbers either, every one of them (none is left from the solve before it)."""
import ctypes

import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.hip import enuc

pytestmark = pytest.mark.gpu

_dp = ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("waters", [1, 3])
def test_nan_in_the_core_hamiltonian(ctx, waters):
    Z, x = M.water_cluster(waters, seed=waters)
    xyz, nocc = M.to_bohr(Z, x), sum(Z) // 2
    ctx.set_system(Z, xyz)
    ctx.eri_build(1e-12)
    S, H = ctx.int1e()
    ctx.rhf(H, S, nocc, enuc(Z, xyz))
    n = ctx.n
    Hn, Sn = np.asfortranarray(H.copy()), np.asfortranarray(S)
    Hn[1, 1] = np.nan
    E, it = ctypes.c_double(0.0), ctypes.c_int(0)
    C, eig = np.zeros((n, n), order="F"), np.zeros(n)
    print(f"[nan] {waters} waters", flush=True)
    rc = ctx.L.myqc_rhf_scf(ctx.h, Hn.ctypes.data_as(_dp), Sn.ctypes.data_as(_dp), nocc, 0.0, None, 1e-10, 1e-8, 3, 0,
                            ctypes.byref(E), C.ctypes.data_as(_dp), eig.ctypes.data_as(_dp), ctypes.byref(it))
    assert rc != 0
    assert np.isnan(E.value) and np.all(np.isnan(eig))
