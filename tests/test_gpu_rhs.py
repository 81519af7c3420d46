"""The cells' right-hand sides (sources at the quadrature points, 16 cells and 32
points at a time, MFMA products with the bases) against the oracle's integration:
more points than a chunk, row counts off the 16-row tiles, a last group of 1, 9
and 16 cells, loads in the flux rows or not, and a non-finite coefficient that
stays with its cell."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_parity import _device_cell_systems, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics,D,k,n,source", [
    ("darcy", 2, 1, 5, 1), ("darcy", 2, 2, 4, 3), ("darcy", 2, 3, 3, 1), ("darcy", 3, 1, 1, 3),
    ("darcy", 3, 2, 3, 1), ("darcy", 3, 3, 2, 3), ("elasticity", 2, 2, 3, 12),
    ("elasticity", 3, 1, 3, 12), ("elasticity", 3, 3, 2, 12)])
def test_cell_rhs_vs_oracle(ctx, physics, D, k, n, source):
    import gridaphybrid as gh
    print(f"cell right-hand sides {physics} D={D} k={k} n={n} source={source}", flush=True)
    nc = n ** D
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, (n,) * D)
    coef = np.random.default_rng(3).uniform(0.2, 0.4, nc)

    def rhs(c):
        if physics == "darcy":
            X = gh.HDGSpaces.darcy_baseline(model, k)
            wf = gh.DarcyHDG(tau=1.0, kappa=c, source=source)
        else:
            X = gh.HDGSpaces.elasticity(model, k)
            wf = gh.ElasticityHDG(tau=1.0, nu=c, E=1.0, source=source)
        op = gh.HybridAffineFEOperator(wf, X, X, [1, 2], [3], ctx=ctx, assemble=False)
        try:
            op.assemble()
        except gh.SingularError:  # (of the cell with the non-finite coefficient)
            assert not np.all(np.isfinite(c))
        b = _device_cell_systems(op, 0, nc)[1][:, :op.info.ni].copy()
        op.close()
        return b

    b = rhs(coef)
    prob = (O.Problem.darcy(D, k, mms=source) if physics == "darcy"
            else O.Problem.elasticity(D, k, tau=1.0, nu=0.3, mms=O.ELAS_MMS_SIN))
    ref = O.hdg_solve(prob, (n,) * D, coef=coef)
    # sums of at most 125 products: the bar of the other integrated blocks
    assert rel(b, ref.b[:, :b.shape[1]]) < 1e-12
    if nc > 1 and source != 1:  # (source 1 does not depend on the coefficient)
        bad = coef.copy()
        bad[nc // 2] = np.nan
        c = rhs(bad)
        rest = np.arange(nc) != nc // 2
        assert np.array_equal(c[rest], b[rest]) and np.isnan(c[nc // 2]).any()
