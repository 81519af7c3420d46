"""Recovery where the flux block is small or large: permeabilities from 1e-8 to 1e8
(Young's moduli of up to 1e8 for elasticity).  The reduced interior block then has entries of the
order of the coefficient beside the functions that no flux sees, which only the
stabilisation holds, and its inverse has to keep both apart.

The recovered values of a cell solve A_ii x = b_i - A_ib lambda; a backward
stable FP64 solve is within a few units of rounding times the condition number of
A_ii, which is the bar (8 eps cond_2) against the solve in extended precision."""
import numpy as np
import pytest

from test_gpu_parity import _device_cell_systems

pytestmark = pytest.mark.gpu


def _solve(A, c):
    """Partial pivoting in extended precision."""
    n = len(c)
    M = np.concatenate([A, c[:, None]], 1).astype(np.longdouble)
    for k in range(n):
        p = k + int(np.argmax(np.abs(M[k:, k])))
        M[[k, p]] = M[[p, k]]
        M[k + 1:, k:] -= np.outer(M[k + 1:, k] / M[k, k], M[k, k:])
    x = np.zeros(n, np.longdouble)
    for k in range(n - 1, -1, -1):
        x[k] = (M[k, n] - M[k, k + 1:n] @ x[k + 1:]) / M[k, k]
    return x


def _check(op, lam, first, cnt):
    """cells first .. first + cnt - 1; boundary traces are zero, or those cells
    have none."""
    nc, na, ni = op.info.ncells, op.info.n_flux, op.info.ni
    fv = op.recover(lam).cpu().numpy()
    x = np.concatenate([fv[:nc * na].reshape(nc, na), fv[nc * na:nc * ni].reshape(nc, ni - na)], 1)
    A, b = _device_cell_systems(op, first, cnt)
    cd = np.asarray(op.cell_blocks()[2]).reshape(nc, -1)[first:first + cnt]
    ld = np.where(cd >= 0, lam[np.maximum(cd, 0)], 0.0).astype(np.longdouble)
    for c in range(cnt):
        rhs = b[c, :ni] - A[c, :ni, ni:] @ ld[c]
        ref = _solve(A[c, :ni, :ni], rhs)
        err = float(np.abs(x[first + c] - ref).max() / np.abs(ref).max())
        cond = np.linalg.cond(A[c, :ni, :ni])
        print(f"  cell {first + c}: error {err:.1e} cond {cond:.1e}", flush=True)
        assert err <= 8 * 2.0 ** -52 * cond


# (D, k, cells, space): a wavefront per cell and 16 cells a workgroup
@pytest.mark.parametrize("D,k,cells,space", [
    (2, 3, (10, 9), 0), (2, 3, (48, 47), 0), (2, 4, (10, 9), 0), (2, 4, (33, 33), 0),
    (3, 1, (5, 5, 4), 0), (3, 1, (13, 13, 13), 0), (3, 2, (4, 4, 4), 0), (3, 3, (3, 3, 3), 0),
    (2, 3, (10, 9), 1), (3, 2, (13, 13, 13), 1)])
@pytest.mark.parametrize("power", [1, -1])
def test_darcy_wide_permeabilities(ctx, D, k, cells, space, power):
    import gridaphybrid as gh
    print(f"wide permeabilities D={D} k={k} cells={cells} space={space} power={power}", flush=True)
    nc = int(np.prod(cells))
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, cells)
    X = gh.HDGSpaces(model, k, k, k, space)
    op = gh.HybridAffineFEOperator(
        gh.DarcyHDG(tau=1.0, kappa=10.0 ** (power * (np.arange(nc) % 9)), source=3), X, X,
        [1, 2], [3], ctx=ctx, assemble=False)
    op.set_family(10)
    op.assemble()
    _check(op, 1 + 0.1 * np.random.default_rng(2).standard_normal(op.info.nfree), nc // 2,
           min(9, nc - nc // 2))
    op.close()


# Darcy's family 8 (both products per cell) and reflected cells, which it serves
@pytest.mark.parametrize("D,k,n", [(2, 3, 9), (3, 1, 5), (3, 2, 4)])
@pytest.mark.parametrize("reflect", [False, True])
def test_darcy_large_permeabilities_products_per_cell(ctx, D, k, n, reflect):
    import gridaphybrid as gh
    import meshgen
    print(f"large permeabilities, family 8, D={D} k={k} reflected={reflect}", flush=True)
    nc = n ** D
    kappa = 10.0 ** (np.arange(nc) % 9)
    if reflect:
        x0, J, cf, nf, perm, _ = meshgen.sheared_rotated_mesh(D, n, seed=14, frac=0.0)
        c, f = nc // 2, (2, 3) if D == 2 else (4, 5)   # xi_0 -> 1 - xi_0
        x0[c] = x0[c] + J[c][:, 0]
        J[c][:, 0] = -J[c][:, 0]
        cf[c][list(f)] = cf[c][list(f[::-1])]
        perm[:] = 0
        perm[c] = [1, 1, 0, 0] if D == 2 else [2, 2, 2, 2, 0, 0]
        model = gh.AffineDiscreteModel(x0=x0, J=J, cell_facets=cf, nfacets=nf, facet_perm=perm)
    else:
        model = gh.CartesianDiscreteModel((0.0, 1.0) * D, (n,) * D)
    X = gh.HDGSpaces.darcy_baseline(model, k)
    op = gh.HybridAffineFEOperator(gh.DarcyHDG(tau=1.0, kappa=kappa, source=0), X, X, [1, 2], [3],
                                   ctx=ctx, assemble=False)
    op.set_family(8)
    op.assemble()
    _check(op, 1 + 0.1 * np.random.default_rng(2).standard_normal(op.info.nfree), nc // 2,
           min(9, nc - nc // 2))
    op.close()


@pytest.mark.parametrize("D,k,E", [(3, 1, 1e4), (3, 1, 1e8), (3, 2, 1e6), (2, 4, 1e8)])
def test_elasticity_large_moduli(ctx, D, k, E):
    import gridaphybrid as gh
    print(f"large modulus D={D} k={k} E={E}", flush=True)
    n = 4 if D == 3 else 5
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, (n,) * D)
    X = gh.HDGSpaces.elasticity(model, k)
    nu = np.random.default_rng(3).uniform(0.2, 0.4, n ** D)
    op = gh.HybridAffineFEOperator(gh.ElasticityHDG(tau=1.0, nu=nu, E=E, source=12), X, X, [1, 2],
                                   [3], ctx=ctx, assemble=False)
    op.set_family(8)
    op.assemble()
    # two interior cells
    _check(op, 1 + 0.1 * np.random.default_rng(2).standard_normal(op.info.nfree),
           21 if D == 3 else 11, 2)
    op.close()
