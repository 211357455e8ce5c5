"""RHF of up to 96 functions from a given density that is not symmetric (its first
Fock build symmetrises it, the later ones take the step's own densities as they
are) ends where the core guess does.  Energies to 1e-8, twice the sum of both
runs' convergence thresholds on the density, whose error they are quadratic in."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.hip import enuc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters", [1, 4, 13])   # 7, 28, 91 functions
def test_unsymmetric_guess(ctx, waters):
    Z, x = M.water_cluster(waters, seed=waters)
    xyz, nocc = M.to_bohr(Z, x), sum(Z) // 2
    print(f"[guess] {waters} waters", flush=True)
    ctx.set_system(Z, xyz)
    ctx.eri_build(1e-12)
    S, H = ctx.int1e()
    r = ctx.rhf(H, S, nocc, enuc(Z, xyz))
    D = ctx.density(r["C"], nocc)
    a = np.random.default_rng(waters).normal(0.0, 1e-3, D.shape)
    g = ctx.rhf(H, S, nocc, enuc(Z, xyz), D_guess=D + a - a.T)
    assert abs(g["E"] - r["E"]) <= 1e-8
