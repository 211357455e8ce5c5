"""The default launch shapes of the stored ERI build: lanes per shell quartet
by the number of quartets of a class, which a shape of -1 lanes restores and
which shapes tuned at another size leave alone.

Helium atoms 15 bohr and more apart make the lanes visible in the last bits:
with the density of one atom j, G_ii is (ii|jj) itself (the charge
distributions of two atoms are screened to nothing, so nothing else is added
to it), and the lanes decide the order of its 81 terms.  Between shapes the
sums agree to rounding: 1e-12 relative to the largest element."""
import numpy as np
import pytest

from myqc_amd import molecules as M

pytestmark = pytest.mark.gpu

RULE = {c: (-1, 256) for c in range(6)}


def _all(lanes):
    return {c: (lanes, 256) for c in range(6)}


@pytest.fixture(autouse=True)
def _rule_afterwards(ctx):
    yield
    ctx.eri_set_shapes(RULE)


def _helium(ctx, count):
    rng = np.random.default_rng(count)
    g = 18.0 * np.array([[x, y, z] for x in range(4) for y in range(4) for z in range(4)], dtype=float)[:count]
    ctx.set_system([2] * count, g + rng.uniform(0.0, 1.7, g.shape))


def _coulomb(ctx):
    """(ii|jj) for the first atoms j, all i != j, of a build at the shapes now in force"""
    n = ctx.n
    ctx.eri_build(0.0)
    out = []
    for j in range(min(n, 6)):
        D = np.zeros((n, n))
        D[j, j] = 1.0
        out.append(np.delete(np.diag(ctx.fock_G(D)), j))
    return np.array(out)


# 231 quartets: eight lanes each; 2.2 million: one (2^18 lanes at most)
@pytest.mark.parametrize("atoms,lanes,other", [(6, 8, 1), (64, 1, 8)])
def test_the_rule_can_be_had_back(ctx, atoms, lanes, other):
    _helium(ctx, atoms)
    print(f"[shapes] {atoms} atoms", flush=True)
    ctx.eri_set_shapes(_all(other))
    b = _coulomb(ctx)
    ctx.eri_set_shapes(_all(lanes))
    a = _coulomb(ctx)
    assert not np.array_equal(a, b)
    ctx.eri_set_shapes(_all(other))
    ctx.eri_set_shapes(RULE)
    assert np.array_equal(_coulomb(ctx), a)


def test_tuned_shapes_stay_with_their_size(ctx):
    ctx.eri_set_shapes(RULE)
    _helium(ctx, 6)
    small = _coulomb(ctx)
    _helium(ctx, 64)
    ctx.eri_build(0.0)
    shapes, _ = ctx.eri_tune(reps=2)
    print(f"[shapes] tuned at 64 atoms: {shapes[0]}", flush=True)
    _helium(ctx, 6)
    assert np.array_equal(_coulomb(ctx), small)


@pytest.mark.parametrize("waters", [1, 24])
def test_rule_against_one_lane(ctx, waters):
    Z, x = M.water_cluster(waters, seed=waters)
    ctx.set_system(Z, M.to_bohr(Z, x))
    n = ctx.n
    D = np.random.default_rng(waters).uniform(-1, 1, (n, n))
    D = D + D.T
    G = []
    for s in (RULE, _all(1)):
        ctx.eri_set_shapes(s)
        ctx.eri_build(1e-12)
        G.append(ctx.fock_G(D))
    assert np.max(np.abs(G[0] - G[1])) <= 1e-12 * np.max(np.abs(G[1]))


def test_other_negative_lanes_are_refused(ctx):
    from myqc_amd.hip import MyqcError
    for sh in ((-2, 256), (3, 256), (8, 32)):
        with pytest.raises(MyqcError):
            ctx.eri_set_shapes({2: sh})
