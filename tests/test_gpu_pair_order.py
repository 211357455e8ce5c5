"""The device's primitive pairs and Schwarz order, where a class has more pairs
than one tile of the ranking kernel holds (1024) and most factors are equal:
helium atoms on a lattice so wide that only (ii|jj) is left, which depends on the
distance alone and comes from the oracle on two atoms.

G of the diagonal density d: G_ii = sum_j d_j (ii|jj) - d_i (ii|ii) / 2, and
nothing off the diagonal.  Tolerance: 1e-12 for each of the terms, which are of order one."""
import numpy as np
import pytest

from myqc_amd.basis import build_basis, read_ftab
from oracle import oracle as O

pytestmark = pytest.mark.gpu

def _coulomb(r):
    Z, x = [2, 2], np.array([[0.0, 0.0, 0.0], [r, 0.0, 0.0]])
    XX = O.eri_full(O.System(Z, x, build_basis(Z), read_ftab()))
    return XX[0, 0, 0, 0], XX[0, 0, 1, 1]

@pytest.mark.parametrize("count", [2, 22, 45, 47, 64])   # 3, 253, 1035, 1128, 2080 pairs
def test_many_equal_pairs(ctx, count):

    g = np.array([[20.0 * x, 20.0 * y, 20.0 * z] for x in range(4) for y in range(4) for z in range(4)])[:count]
    Z = [2] * count
    print(f"[pairs] {count} atoms", flush=True)
    ctx.set_system(Z, g)
    n2 = np.rint(((g[:, None] - g[None]) ** 2).sum(-1) / 400.0).astype(int)
    V = {k: _coulomb(20.0 * np.sqrt(k))[1] for k in np.unique(n2) if k}
    V[0] = _coulomb(20.0)[0]
    C = np.vectorize(V.get)(n2)
    d = np.random.default_rng(count).uniform(0.5, 2.0, count)
    assert ctx.eri_build(0.0) == count * (count + 1) * (count * (count + 1) // 2 + 1) // 4
    G = ctx.fock_G(np.diag(d))
    ref = np.diag(C @ d - 0.5 * d * np.diag(C))
    assert np.max(np.abs(G - ref)) <= 1e-12 * count
