"""Dense integrals at the sizes where their expansion changes form
(csrc/dense.hip): a block in 16 KiB of LDS (n <= 63), in 128 KiB (n <= 180), in
several ranges of u above; the dense array in one piece (n <= 80) or in slabs.

An integral depends on its own shells alone, so those of a few of the atoms are
compared with the CPU oracle's for these atoms.  Tolerance: the parity bound of
the integrals, 1e-10 (they agree to a few 1e-15).  The eight places of a value
are equal bit for bit."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.basis import build_basis, read_ftab
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FT = read_ftab()


def _system(ctx, n):
    """n functions: waters and helium atoms; (Z, xyz, first function of each atom)"""
    w, he = divmod(n, 7)
    Z, x = M.water_cluster(w, seed=n, box=12.0 * (w / 40.0) ** (1 / 3) + 0.5)
    Z = list(Z) + [2] * he
    xyz = np.concatenate([M.to_bohr(Z[:3 * w], x), np.array([[-5.0, 4.0 * k, 0.0] for k in range(he)]).reshape(-1, 3)])
    ctx.set_system(Z, xyz)
    assert ctx.n == n
    return Z, xyz, np.cumsum([0] + [5 if z == 8 else 1 for z in Z])


def _some_atoms(Z, xyz, first, atoms):
    """functions of these atoms, and the oracle's integrals over them"""
    z, x = [Z[a] for a in atoms], xyz[atoms]
    f = np.concatenate([np.arange(first[a], first[a + 1]) for a in atoms])
    return f, O.eri_full(O.System(z, x, build_basis(z), FT))


@pytest.mark.parametrize("n", [62, 63, 64, 80, 81, 98])
def test_dense_array_at_size_edges(ctx, n):
    Z, xyz, first = _system(ctx, n)
    print(f"[dense] n = {n}", flush=True)
    XX = ctx.eri_full(0.0)
    for p in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(XX, XX.transpose(p))
    last = len(Z) - 1
    for atoms in ([0, 1, last], [0, 3, last - 1], [last - 2, 12, 5]):
        f, want = _some_atoms(Z, xyz, first, atoms)
        assert np.max(np.abs(XX[np.ix_(f, f, f, f)] - want)) <= 1e-10


@pytest.mark.parametrize("n", [62, 63, 64, 180, 181])
def test_transform_blocks_at_size_edges(ctx, n):
    """(ia|jb) over orbitals that are single functions"""
    Z, xyz, first = _system(ctx, n)
    print(f"[blocks] n = {n}", flush=True)
    atoms = [0, 1, 36 if n > 100 else 12, len(Z) - 1]
    f, want = _some_atoms(Z, xyz, first, atoms)
    o = 5                                     # occupied: the functions of the first atom
    perm = np.concatenate([f, np.setdiff1d(np.arange(n), f)])
    t = ctx.ao2mo(np.eye(n)[:, perm], o)      # no build stored: unscreened integrals
    m = len(f)
    assert np.max(np.abs(t[:, :m - o, :, :m - o] - want[:o, o:m, :o, o:m])) <= 1e-10
