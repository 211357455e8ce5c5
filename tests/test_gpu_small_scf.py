"""The one-launch SCF step of small systems (csrc/scf_small.hip) at the sizes
where its 16-wide tiles, its thread counts and its limit (96 functions) change,
against the equations the result has to satisfy, written with the library's
own integrals and Fock build (pinned by the parity tests).

Tolerances: the loop converges max|dD| to 1e-8 with the commutator's norm below
1e-6, so F C = S C e holds to 1e-6 in each element (|C| <= 2); the orbitals are
rotations of X applied to machine precision (1e-10); two converged runs agree
in energy to the parity bound, 1e-8 Eh."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.hip import FP32, FP64, enuc

pytestmark = pytest.mark.gpu


def _cluster(n):
    """n functions: n // 7 waters and n % 7 helium atoms 3 A apart beside them."""
    w, h = divmod(n, 7)
    Z, x = ([], np.zeros((0, 3))) if w == 0 else M.water_cluster(w, seed=n, box=12.0 * (w / 40.0) ** (1 / 3) + 0.5)
    x = np.concatenate([x, [[-4.0, 3.0 * k, 0.0] for k in range(h)]]) if h else x
    Z = list(Z) + [2] * h
    return Z, M.to_bohr(Z, x), 5 * w + h


def _check(ctx, r, S, H, nocc, e_nuc):
    C, e = r["C"], r["eig"]
    D = 2 * C[:, :nocc] @ C[:, :nocc].T
    G = ctx.fock_G(D)
    F = H + G
    assert np.max(np.abs(C.T @ S @ C - np.eye(len(e)))) <= 1e-10
    assert np.max(np.abs(F @ C - S @ C * e)) <= 1e-6
    assert np.all(np.diff(e) >= 0)
    assert abs(0.5 * np.sum(D * (F + H)) + e_nuc - r["E"]) <= 1e-8


@pytest.mark.parametrize("n", [1, 2, 7, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 81, 95, 96, 97])
def test_solution_at_tile_edges(ctx, n):
    Z, xyz, nocc = _cluster(n)
    ctx.set_system(Z, xyz)
    assert ctx.n == n
    S, H = ctx.int1e()
    ctx.eri_build(1e-12)
    en = enuc(Z, xyz)
    r = ctx.rhf(H, S, nocc, en)
    _check(ctx, r, S, H, nocc, en)
    m = ctx.rhf(H, S, nocc, en, precision=FP32)
    _check(ctx, m, S, H, nocc, en)
    assert abs(m["E"] - r["E"]) <= 1e-8
    # restarts from the orbitals and from the density converge at once
    for kw in (dict(C_guess=r["C"]), dict(D_guess=ctx.density(r["C"], nocc))):
        q = ctx.rhf(H, S, nocc, en, precision=FP64, **kw)
        assert abs(q["E"] - r["E"]) <= 1e-8 and q["iterations"] <= 4


def test_empty_and_full_occupation(ctx):
    Z, xyz, _ = _cluster(14)
    ctx.set_system(Z, xyz)
    S, H = ctx.int1e()
    ctx.eri_build(1e-12)
    for nocc in (0, 14):
        r = ctx.rhf(H, S, nocc, 0.0)
        _check(ctx, r, S, H, nocc, 0.0)
        assert r["purifications"] == 0


def test_unconverged_run_reports(ctx):
    from myqc_amd.hip import MyqcError
    Z, xyz, nocc = _cluster(28)
    ctx.set_system(Z, xyz)
    S, H = ctx.int1e()
    ctx.eri_build(1e-12)
    with pytest.raises(MyqcError, match="did not converge in 3"):
        ctx.rhf(H, S, nocc, enuc(Z, xyz), max_iter=3)


def test_singular_overlap_is_refused(ctx):
    from myqc_amd.hip import MyqcError
    Z, xyz, nocc = _cluster(14)
    ctx.set_system(Z, xyz)
    S, H = ctx.int1e()
    ctx.eri_build(1e-12)
    S = S.copy()
    S[1] = S[0]
    S[:, 1] = S[:, 0]
    with pytest.raises(MyqcError, match="singular"):
        ctx.rhf(H, S, nocc, enuc(Z, xyz))


@pytest.mark.parametrize("n,kappa", [(14, 1e3), (30, 1e6), (60, 1e5), (90, 1e8)])
def test_ill_conditioned_overlap(ctx, n, kappa):
    """An S of condition number kappa: the orbitals stay S-orthonormal.
    Tolerance: X = S^-1/2 from products carries an error of order kappa eps in
    X S X - I (1e-16 kappa), with a factor 1e3 for n and the steps."""
    Z, xyz, _ = _cluster(n)
    ctx.set_system(Z, xyz)
    S, H = ctx.int1e()
    ctx.eri_build(1e-12)
    w, U = np.linalg.eigh(S)
    w = np.exp(np.linspace(-np.log(kappa), 0.0, n))
    Sx = (U * w) @ U.T
    Sx = 0.5 * (Sx + Sx.T)
    Q = (U * np.sqrt(w)) @ U.T
    Hx = Q @ np.diag(np.linspace(-20.0, 1.0, n)) @ Q
    # no electrons: F = H, and the run ends at once (with electrons D grows as
    # kappa, and no run brings |dE| below 1e-10 of such an energy)
    C = ctx.rhf(0.5 * (Hx + Hx.T), Sx, 0, 0.0)["C"]
    assert np.max(np.abs(C.T @ Sx @ C - np.eye(n))) <= 1e-13 * kappa
