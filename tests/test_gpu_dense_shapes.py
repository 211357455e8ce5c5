"""Dense integrals and transforms do not follow the launch shapes that a stored
build was given: other lanes per quartet sum its primitive quartets in another
order, and the dense results stay those of the shapes by the rule, bit for bit,
whether or not integrals are stored at their threshold."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.hip import BF16X3, Context

pytestmark = pytest.mark.gpu

RULE = {c: (-1, 256) for c in range(6)}
TOL = 1e-12


def _results(ctx, nocc):
    n = ctx.n
    C = np.linalg.qr(np.random.default_rng(n).normal(size=(n, n)))[0]
    return [ctx.eri_full(TOL), ctx.ao2mo(C, nocc), ctx.ao2mo(C, nocc, BF16X3),
            *ctx.ao2mo_uhf(C, C[:, ::-1], nocc, nocc - 1).values()]


@pytest.mark.parametrize("waters,lanes", [(1, 1), (4, 1), (4, 2)])
def test_dense_results_do_not_follow_given_shapes(ctx, waters, lanes):
    Z, x = M.water_cluster(waters, seed=waters, box=3.0 + waters)
    xyz, nocc = M.to_bohr(Z, x), sum(Z) // 2
    print(f"[dense] {waters} waters, {lanes} lanes", flush=True)
    try:
        with Context(0) as c:
            c.set_system(Z, xyz)
            c.eri_build(TOL)   # (the threshold of the transforms)
            want = _results(c, nocc)
        ctx.eri_set_shapes({c: (lanes, 64) for c in range(6)})
        ctx.set_system(Z, xyz)
        stored = ctx.eri_build(TOL)
        D = np.eye(ctx.n)
        G = ctx.fock_G(D)
        for a, b in zip(_results(ctx, nocc), want):
            assert np.array_equal(a, b)
        # the given build is still the stored one
        assert np.max(np.abs(ctx.fock_G(D) - G)) <= 1e-13 * np.max(np.abs(G))
        # nor those a tune leaves in the store
        ctx.eri_tune(reps=1)
        for a, b in zip(_results(ctx, nocc), want):
            assert np.array_equal(a, b)
        ctx.eri_set_shapes(RULE)
        assert ctx.eri_build(TOL) == stored
        for a, b in zip(_results(ctx, nocc), want):
            assert np.array_equal(a, b)
    finally:
        ctx.eri_set_shapes(RULE)
