"""The flux families where the orders of the three fields differ (np and nq on
either side of a row tile, one potential function, no function unseen by the
flux): against the dense elimination of the same cells, S and g to 1e-12, the
recovered values to 1e-11 (the bars of the other comparisons of two families)."""
import numpy as np
import pytest

from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("physics,D,space,orders,cells", [
    ("darcy", 2, 0, (2, 1, 2), (7, 5)), ("darcy", 2, 0, (2, 3, 2), (7, 5)),
    ("darcy", 2, 0, (2, 3, 2), (48, 43)), ("darcy", 2, 0, (4, 3, 3), (36, 29)),
    ("darcy", 2, 0, (3, 4, 3), (36, 29)), ("darcy", 2, 1, (1, 0, 1), (50, 41)),
    ("darcy", 2, 1, (3, 2, 3), (6, 5)), ("darcy", 3, 0, (1, 0, 1), (13, 13, 13)),
    ("darcy", 3, 0, (2, 1, 1), (4, 4, 3)), ("darcy", 3, 0, (1, 2, 1), (4, 4, 3)),
    ("elasticity", 2, 0, (2, 2, 2), (5, 4)), ("elasticity", 2, 1, (1, 1, 1), (5, 4)),
    ("elasticity", 3, 1, (2, 2, 2), (3, 3, 2)), ("elasticity", 3, 1, (1, 2, 2), (3, 3, 2))])
def test_orders_that_differ(ctx, physics, D, space, orders, cells):
    import gridaphybrid as gh
    print(f"{physics} D={D} space={space} orders={orders} cells={cells}", flush=True)
    nc = int(np.prod(cells))
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, cells)
    X = gh.HDGSpaces(model, *orders, space)
    coef = np.random.default_rng(4).uniform(0.2, 0.4, nc)
    if physics == "darcy":
        wf, flux = gh.DarcyHDG(tau=1.0, kappa=coef, source=3), 10
    else:
        wf, flux = gh.ElasticityHDG(tau=4.0, nu=coef, E=1.0, source=12), 8
    op = gh.HybridAffineFEOperator(wf, X, X, [1, 2], [3], ctx=ctx, assemble=False)
    lam = np.random.default_rng(5).standard_normal(op.info.nfree)
    out = []
    n = op.info.ni + op.info.nb
    for family in (flux, 1 if n < 72 else 5 if n <= 256 else 4):
        op.set_family(family)
        op.assemble()
        assert op.factor_rows()[1] == family
        S, g, _ = op.cell_blocks()
        out.append((S, g, op.recover(lam).cpu().numpy()))
    for a, b, tol in zip(out[0], out[1], (1e-12, 1e-12, 1e-11)):
        assert rel(a, b) < tol
    op.close()
