"""Darcy's flux recovery of 16 cells per workgroup against the direct solve of
each cell's interior system: one to four row tiles, np and nq off the tile and
off the k-step, a last group of 1, 15 and 16 cells, and a non-finite trace."""
import numpy as np
import pytest

from test_gpu_parity import _device_cell_systems, rel

pytestmark = pytest.mark.gpu

REF = 10
# (D, k, cells): np = nq = (k + 1)^D
CASES = [(2, 1, (64, 33)), (2, 2, (683, 3)), (2, 3, (23, 91)), (2, 4, (5, 5)),
         (3, 1, (13, 13, 13)), (3, 2, (1, 1, 1)), (3, 2, (3, 3, 7)), (3, 2, (17, 16, 16)),
         (3, 3, (4, 2, 2)), (3, 3, (31, 1, 1))]


@pytest.mark.parametrize("D,k,cells", CASES)
def test_group_recovery_vs_direct_solve(ctx, D, k, cells):
    import gridaphybrid as gh
    print(f"group recovery D={D} k={k} cells={cells}", flush=True)
    rng = np.random.default_rng(5)
    nc = int(np.prod(cells))
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, cells)
    X = gh.HDGSpaces.darcy_baseline(model, k)
    op = gh.HybridAffineFEOperator(
        gh.DarcyHDG(tau=1.0, kappa=rng.uniform(0.5, 2.0, nc), source=3), X, X, [1, 2], [3],
        ctx=ctx, assemble=False)
    op.set_family(REF)
    op.assemble()
    na, ni, nfree = op.info.n_flux, op.info.ni, op.info.nfree
    assert op.factor_rows() == (ni - na, REF)
    lam = rng.standard_normal(nfree)
    fv = op.recover(lam).cpu().numpy()
    first = max(0, nc - 40)  # the last groups, whole and partial
    A, b = _device_cell_systems(op, first, nc - first)
    _, _, cd = op.cell_blocks()
    cd = np.asarray(cd).reshape(nc, -1)
    ld = _trace_values(op, lam, cd[first:])
    c = b[:, :ni] - np.einsum("cij,cj->ci", A[:, :ni, ni:], ld)
    x = np.linalg.solve(A[:, :ni, :ni], c[..., None])[..., 0]
    got = np.concatenate([fv[:nc * na].reshape(nc, na),
                          fv[nc * na:nc * ni].reshape(nc, ni - na)], 1)
    # the bar of the other comparisons of two recoveries
    assert rel(got[first:], x) < 1e-11
    # a non-finite trace value stays with the cells of its facet
    if nfree:
        bad = lam.copy()
        bad[nfree // 2] = np.nan
        fb = op.recover(bad).cpu().numpy()
        gb = np.concatenate([fb[:nc * na].reshape(nc, na),
                             fb[nc * na:nc * ni].reshape(nc, ni - na)], 1)
        hit = (cd == nfree // 2).any(1)
        assert hit.any() and np.isnan(gb[hit]).any(1).all()
        assert np.array_equal(gb[~hit], got[~hit])
    op.close()


def _trace_values(op, lam, cd):
    """lambda of the cells' boundary columns (homogeneous boundary values)."""
    v = np.zeros(cd.shape)
    v[cd >= 0] = lam[cd[cd >= 0]]
    return v
