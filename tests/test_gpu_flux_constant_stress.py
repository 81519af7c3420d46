"""The flux elimination (family 8) with piecewise constant stresses: the block
between stresses and displacement is empty, so its transpose symmetry has no
sign.  The family is accepted as for every other order and agrees with the dense
elimination of the same cells: S and g to 1e-12, the recovered values to 1e-11
(the bars of the other comparisons of two families)."""
import numpy as np
import pytest

from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,space,orders", [
    (2, "P", (0, 1, 1)), (2, "Q", (0, 0, 0)), (3, "P", (0, 1, 0)), (3, "Q", (0, 1, 1))])
def test_constant_stress_flux_family(ctx, D, space, orders):
    import gridaphybrid as gh
    print(f"constant stresses D={D} space={space} orders={orders}", flush=True)
    n = 3
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, (n,) * D)
    X = gh.HDGSpaces(model, *orders, gh.SPACE_Q if space == "Q" else gh.SPACE_P)
    nu = np.random.default_rng(4).uniform(0.2, 0.4, n ** D)
    wf = gh.ElasticityHDG(tau=float(n), nu=nu, E=1.0, source=12)
    op = gh.HybridAffineFEOperator(wf, X, X, [1, 2], [3], ctx=ctx, assemble=False)
    lam = np.random.default_rng(5).standard_normal(op.info.nfree)
    out = []
    for family in (8, 1 if op.info.ni + op.info.nb < 72 else 5):
        op.set_family(family)
        op.assemble()
        assert op.factor_rows()[1] == family
        S, g, _ = op.cell_blocks()
        out.append((S, g, op.recover(lam).cpu().numpy()))
    for a, b, tol in zip(out[0], out[1], (1e-12, 1e-12, 1e-11)):
        assert rel(a, b) < tol
    if op.info.ni + op.info.nb > 96:
        op.set_family(None)
        op.assemble()
        assert op.factor_rows()[1] == 8  # the class's default
    op.close()
