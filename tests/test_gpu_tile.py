"""The tile elimination (blocked LU of the interior block in LDS, the boundary
products on FP64 MFMA tiles) at the edges of its tiles and strips.

Map level: interior sizes around the 16-row tiles and the 32, 64, 112 and 128
row limits, boundary sizes around the 16-column strips and the limits of one
strip per wavefront, against the oracle's LAPACK-order condensation.  The
matrices are standard normal plus n I, cond(A_ii) below 10, so two FP64
eliminations agree to a few n eps ~ 1e-13: the bar is 1e-12.

Operator level: elasticity from the reference products on sheared cells, one of
them reflected (det J < 0), against the oracle's integration, with the bar of
the existing elasticity tests (ten times the oracle's own self-variation, at
least 1e-12)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("ni,nb", [
    (1, 71), (16, 63), (17, 56), (31, 63), (32, 64), (33, 47), (63, 111), (64, 127), (65, 15),
    (80, 0), (96, 191), (112, 160), (113, 16), (127, 127), (128, 1)])
def test_tile_map_sizes(ctx, ni, nb):
    import gridaphybrid as gh
    print(f"tile map ni={ni} nb={nb}", flush=True)
    rng = np.random.default_rng(1000 * ni + nb)
    nc, n = 5, ni + nb
    A = rng.standard_normal((nc, n, n)) + n * np.eye(n)[None]
    # a pivot away from the diagonal in every column of every other cell
    A[::2, :ni] = A[::2, np.r_[1:ni, 0]]
    b = rng.standard_normal((nc, n))
    if nb:
        S, g = gh.StaticCondensationMap([1], [2], ctx).evaluate(A, b, [ni, nb])
        So, go, info = O.condense(A, b, ni, nb)
        assert not info.any()
        assert rel(S.cpu().numpy(), So) < RTOL and rel(g.cpu().numpy(), go) < RTOL
    else:
        nb, A, b = 1, np.pad(A, ((0, 0), (0, 1), (0, 1))), np.pad(b, ((0, 0), (0, 1)))
    x = rng.standard_normal((nc, nb))
    xi, _ = gh.BackwardStaticCondensationMap([1], [2], ctx).evaluate(A, b, x, [ni, nb])
    xo, _ = O.recover(A, b, x, ni, nb)
    assert rel(xi.cpu().numpy(), xo) < RTOL


def test_tile_singular_and_nonfinite_cells_stay_alone(ctx):
    """A singular cell reports its first zero pivot (getrf info), a cell with an
    infinity or a NaN its own non-finite result; the others keep their values."""
    import gridaphybrid as gh
    rng = np.random.default_rng(5)
    ni, nb, nc = 60, 30, 6
    A = rng.standard_normal((nc, ni + nb, ni + nb)) + 90 * np.eye(ni + nb)[None]
    b = rng.standard_normal((nc, ni + nb))
    good = [0, 2, 5]
    So, go, _ = O.condense(A[good], b[good], ni, nb)
    A[1, :ni, 20] = 0.0
    A[3, 7, 9] = np.inf
    A[4, 70, 3] = np.nan
    S, g, info = gh.StaticCondensationMap([1], [2], ctx).evaluate(A, b, [ni, nb],
                                                                 return_info=True)
    S, g, info = S.cpu().numpy(), g.cpu().numpy(), info.cpu().numpy()
    assert info[1] == 21 and not info[good].any()
    assert rel(S[good], So) < RTOL and rel(g[good], go) < RTOL
    assert not np.isfinite(S[3]).all() and not np.isfinite(S[4]).all()


@pytest.mark.parametrize("D,k,reflect", [(2, 2, True), (3, 1, False), (3, 2, False), (3, 3, False)])
def test_elasticity_reference_products(ctx, D, k, reflect):
    import gridaphybrid as gh
    import meshgen
    print(f"elasticity from reference products D={D} k={k} reflected={reflect}", flush=True)
    n = 2
    x0, J, cf, nf, perm, _ = meshgen.sheared_rotated_mesh(D, n, seed=21, frac=0.0)
    if reflect:  # 2D: xi_0 -> 1 - xi_0 in the last cell, facets 2 and 3 swap, 0 and 1 flip
        x0[3] = x0[3] + J[3][:, 0]
        J[3][:, 0] = -J[3][:, 0]
        cf[3][[2, 3]] = cf[3][[3, 2]]
        perm[3] = [1, 1, 0, 0]
    fperm = perm if perm.any() else None
    nu = np.random.default_rng(22).uniform(0.2, 0.4, n ** D)
    model = gh.AffineDiscreteModel(x0=x0, J=J, cell_facets=cf, nfacets=nf, facet_perm=fperm)
    X = gh.HDGSpaces.elasticity(model, k)
    op = gh.HybridAffineFEOperator(gh.ElasticityHDG(tau=float(n), nu=nu, E=1.0, source=12), X, X,
                                   [1, 2], [3], ctx=ctx, assemble=False)
    op.set_family(8)
    op.assemble()
    assert op.factor_rows() == (op.info.ni - op.info.n_flux, 8)
    ref = O.hdg_solve_mesh(O.Problem.elasticity(D, k, tau=float(n), nu=0.3, mms=O.ELAS_MMS_SIN),
                           meshgen.oracle_mesh(x0, J, cf, nf, fperm), coef=nu)
    ni, nb = op.info.ni, op.info.nb
    p = np.r_[np.random.default_rng(1).permutation(ni), ni:ni + nb]
    S2, g2, _ = O.condense(ref.A[:, p][:, :, p], ref.b[:, p], ni, nb)
    S, g, cd = op.cell_blocks()
    assert np.array_equal(cd, ref.cell_dofs)
    assert rel(S, ref.S) < max(RTOL, 10 * rel(S2, ref.S))
    assert rel(g, ref.g) < max(RTOL, 10 * rel(g2, ref.g))
    fv = op.recover(ref.lam).cpu().numpy()
    assert rel(fv, ref.free_values) < (1e-9 if k == 3 else 1e-11)
    op.close()
