"""The batched SCF kernel at the edges of its size classes (16, 32, 40 functions,
a wavefront's rows and tiles, one function, all levels occupied) against the
single-molecule path, and its refusals.

Tolerances: energies 1e-8, as the batch is pinned elsewhere; both paths stop at
density changes below 1e-8 with errors a small factor above that, so their
densities agree to 1e-7."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.basis import build_basis
from myqc_amd.hip import enuc

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 15, 16, 17, 24, 25, 31, 32, 33, 36, 37, 39, 40]


def _molecule(n):
    """waters and, off to the side, helium atoms: n functions"""
    w, he = divmod(n, 7)
    Z, x = M.water_cluster(w, seed=n) if w else ([], np.zeros((0, 3)))
    x = M.to_bohr(Z, x) if w else x
    far = np.array([[40.0 + 4.0 * k, 0.5 * k, 0.0] for k in range(he)]).reshape(-1, 3)
    return list(Z) + [2] * he, np.concatenate([np.asarray(x), far])


@pytest.fixture(scope="module")
def solved(ctx):
    mols = [_molecule(n) for n in SIZES]
    ctx.batch_set(mols)
    E, it, cv = ctx.batch_rhf(e_tol=1e-10, d_tol=1e-8, max_iter=100)
    return mols, E, cv, ctx.batch_density()


@pytest.mark.parametrize("k", range(len(SIZES)), ids=[str(n) for n in SIZES])
def test_batch_size(ctx, solved, k):
    mols, E, cv, D = solved
    Z, xyz = mols[k]
    assert build_basis(Z).norb == SIZES[k] and cv[k] == 1
    print(f"[batch] n = {SIZES[k]}", flush=True)
    ctx.set_system(Z, xyz)
    ctx.eri_build(0.0)
    S, H = ctx.int1e()
    r = ctx.rhf(H, S, sum(Z) // 2, enuc(Z, xyz), e_tol=1e-10, d_tol=1e-8, max_iter=100)
    assert abs(E[k] - r["E"]) <= 1e-8
    assert np.max(np.abs(D[k] - ctx.density(r["C"], sum(Z) // 2))) <= 1e-7


def test_batch_guess_need_not_be_symmetric(ctx):
    # the densities of the solution with an antisymmetric part converge to it again
    mols = [_molecule(n) for n in (7, 17, 33)]
    ctx.batch_set(mols)
    E, _, cv = ctx.batch_rhf(e_tol=1e-10, d_tol=1e-8, max_iter=100)
    rng = np.random.default_rng(1)
    G = []
    for d in ctx.batch_density():
        a = rng.normal(0.0, 1e-3, d.shape)
        G.append(d + a - a.T)
    E1, _, cv1 = ctx.batch_rhf(D_guess=G, e_tol=1e-10, d_tol=1e-8, max_iter=100)
    assert np.all(cv == 1) and np.all(cv1 == 1)
    assert np.max(np.abs(E1 - E)) <= 1e-8


@pytest.mark.parametrize("d,conv", [(1e-6, -1), (1e-3, 1)])
def test_batch_near_singular_overlap(ctx, d, conv):
    # two hydrogens at d: the smaller overlap eigenvalue is of the order of d^2 / 5
    Z, x = M.water_cluster(1, seed=3)
    x = np.asarray(M.to_bohr(Z, x))
    pair = np.array([[30.0, 0.0, 0.0], [30.0 + d, 0.0, 0.0]])
    ctx.batch_set([(list(Z) + [1, 1], np.concatenate([x, pair])), (Z, x)])
    E, _, cv = ctx.batch_rhf(e_tol=1e-10, d_tol=1e-8, max_iter=100)
    assert cv[1] == 1
    assert (cv[0] == -1) == (conv == -1)
