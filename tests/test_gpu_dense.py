"""Dense integrals expanded from the stored ones (csrc/dense.hip): sizes at the
edges of the 32-wide tiles, systems without one or two of the pair classes,
and what the call leaves behind, against the CPU oracle and the symmetries.

Tolerance: the parity bound of the integrals, 1e-10 (they agree to a few
1e-15; the expansion multiplies by powers of two only)."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.basis import build_basis, read_ftab
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _helium(k, seed):
    rng = np.random.default_rng(seed)
    return [2] * k, rng.uniform(0.0, 3.0 * k ** (1.0 / 3.0), (k, 3))


@pytest.mark.parametrize("Z,xyz", [
    _helium(1, 0), _helium(2, 1),                    # one class of pairs, n = 1 and 2
    ([1, 9], np.array([[0, 0, 0], [0, 0, 0.92]])),
    M.random_molecule(np.random.default_rng(4)),
    tuple(np.concatenate(p) if k else list(p[0]) + list(p[1])
          for k, p in enumerate(zip(M.water_cluster(4, 9, 6.0), _helium(3, 2)))),   # n = 31
    tuple(np.concatenate(p) if k else list(p[0]) + list(p[1])
          for k, p in enumerate(zip(M.water_cluster(4, 9, 6.0), _helium(4, 3)))),   # n = 32
    tuple(np.concatenate(p) if k else list(p[0]) + list(p[1])
          for k, p in enumerate(zip(M.water_cluster(4, 9, 6.0), _helium(5, 4)))),   # n = 33
])
def test_dense_integrals_at_tile_edges(ctx, Z, xyz):
    x = M.to_bohr(Z, xyz)
    basis, ftab = build_basis(list(Z)), read_ftab()
    ctx.set_system(Z, x, basis, ftab)
    XX = ctx.eri_full(0.0)
    for p in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(XX, XX.transpose(p))
    assert np.max(np.abs(XX - O.eri_full(O.System(Z, x, basis, ftab)))) <= 1e-10


def test_blocks_in_several_ranges(ctx):
    """27 waters (n = 189): a block no longer fits one workgroup's LDS.  The
    transform's (ia|jb) for orbitals that are single functions are the
    integrals themselves, compared with the Fock build of one density
    element, G(j,b) for D at (i,a).  Tolerance 1e-10 as above."""
    Z, x = M.water_cluster(27, 5, 10.6)
    xyz = M.to_bohr(Z, x)
    ctx.set_system(Z, xyz)
    n = ctx.n
    assert n == 189
    perm = np.random.default_rng(6).permutation(n)
    C, o = np.eye(n)[:, perm], 4
    ctx.eri_build(1e-13)
    t = ctx.ao2mo(C, o)                            # (ia|jb), i, j of the first four functions of perm
    for i in range(o):
        for a in (0, 57, 180):
            D = np.zeros((n, n))
            D[perm[i], perm[o + a]] = D[perm[o + a], perm[i]] = 0.5
            J = ctx.fock_G_uhf(D, D)[0]          # 2 J[D] - K[D]
            K = -ctx.fock_G_uhf(D, -D)[0]          # K[D]
            Jd = (J + K) / 2
            want = Jd[np.ix_(perm[:o], perm[o:])]
            assert np.max(np.abs(t[i, a] - want)) <= 1e-10


def test_dense_call_keeps_the_stored_integrals(ctx):
    Z, x = M.water_cluster(5, 3, 8.0)
    xyz = M.to_bohr(Z, x)
    ctx.set_system(Z, xyz)
    n = ctx.n
    D = np.random.default_rng(1).uniform(-1, 1, (n, n))
    D = D + D.T
    ns = ctx.eri_build(1e-9)
    G = ctx.fock_G(D)
    full = ctx.eri_full(0.0)                       # another threshold than the stored build's
    assert np.max(np.abs(ctx.fock_G(D) - G)) <= 1e-12 * np.max(np.abs(G))
    same = ctx.eri_full(1e-9)                      # the stored build itself, screened
    assert np.max(np.abs(same - full)) <= 2e-9
    assert np.count_nonzero(same) <= np.count_nonzero(full)
    assert ctx.eri_build(1e-9) == ns


def test_dense_call_does_not_stand_in_for_a_build():
    from myqc_amd.hip import Context, MyqcError
    with Context(0) as c:
        Z, x = M.water()
        c.set_system(Z, M.to_bohr(Z, x))
        c.eri_full(0.0)
        with pytest.raises(MyqcError):
            c.fock_G(np.eye(c.n))
        c.ao2mo(np.eye(c.n), 5)
        with pytest.raises(MyqcError):
            c.fock_G(np.eye(c.n))


def test_transform_over_several_chunks(ctx):
    """15 waters (n = 105: 5565 blocks, two chunks at the buffer's bound) in
    FP64 against the dense array's own contraction.  Tolerance: the record
    bound of the transform, 1e-10."""
    Z, x = M.water_cluster(15, 7, 9.0)
    xyz = M.to_bohr(Z, x)
    ctx.set_system(Z, xyz)
    n = ctx.n
    C = np.linalg.qr(np.random.default_rng(2).normal(size=(n, n)))[0]
    o = 75
    t = ctx.ao2mo(C, o)
    XX = ctx.eri_full(0.0).reshape(n * n, n * n, order="F")
    rng = np.random.default_rng(3)
    for _ in range(12):
        i, j, a, b = rng.integers(o), rng.integers(o), rng.integers(n - o), rng.integers(n - o)
        L = np.outer(C[:, i], C[:, o + a]).ravel(order="F")
        R = np.outer(C[:, j], C[:, o + b]).ravel(order="F")
        assert abs(t[i, a, j, b] - L @ XX @ R) <= 1e-10
