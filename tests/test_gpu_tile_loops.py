"""The tile elimination where its workgroups take several cells, and the 65 to 80
row interiors.

A launch has at most 256 workgroups per CU slot, so the cells beyond the first
grid reuse the LDS (factors, row moves, reciprocals, staged Y) of the cells
before them: singular, infinite and NaN cells sit in the first pass, and every
cell has to give, bit for bit, what the same cell gives in a call of its own.

Sizes: the matrices are standard normal plus n I, cond(A_ii) below 10, so two
FP64 eliminations agree to a few n eps ~ 1e-13: the bar is 1e-12."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_tile import rel

pytestmark = pytest.mark.gpu

RTOL = 1e-12


@pytest.mark.parametrize("ni,nb", [
    (65, 7), (66, 48), (72, 20), (79, 111), (80, 16), (80, 127), (81, 33)])
def test_interiors_of_65_to_80_rows(ctx, ni, nb):
    import gridaphybrid as gh
    print(f"tile map ni={ni} nb={nb}", flush=True)
    rng = np.random.default_rng(1000 * ni + nb)
    nc, n = 5, ni + nb
    A = rng.standard_normal((nc, n, n)) + n * np.eye(n)[None]
    A[::2, :ni] = A[::2, np.r_[1:ni, 0]]  # a pivot away from the diagonal
    b = rng.standard_normal((nc, n))
    S, g = gh.StaticCondensationMap([1], [2], ctx).evaluate(A, b, [ni, nb])
    So, go, info = O.condense(A, b, ni, nb)
    assert not info.any()
    assert rel(S.cpu().numpy(), So) < RTOL and rel(g.cpu().numpy(), go) < RTOL
    x = rng.standard_normal((nc, nb))
    xi, _ = gh.BackwardStaticCondensationMap([1], [2], ctx).evaluate(A, b, x, [ni, nb])
    xo, _ = O.recover(A, b, x, ni, nb)
    assert rel(xi.cpu().numpy(), xo) < RTOL


# (ni, nb, cells): 2,048 workgroups up to 80 rows, 1,024 beyond, 12,288 wavefronts
@pytest.mark.parametrize("ni,nb,nc", [
    (27, 54, 12400), (14, 60, 12400), (60, 30, 2150), (72, 20, 2150), (100, 40, 1100),
    (120, 30, 1100)])
def test_cells_after_a_bad_cell_in_the_same_workgroup(ctx, ni, nb, nc):
    import gridaphybrid as gh
    import torch
    print(f"tile loops ni={ni} nb={nb} cells={nc}", flush=True)
    rng = np.random.default_rng(ni)
    n, nd = ni + nb, 9
    A = rng.standard_normal((nd, n, n)) + n * np.eye(n)[None]
    A[::2, :ni] = A[::2, np.r_[1:ni, 0]]
    b = rng.standard_normal((nd, n))
    A[6, :ni, ni // 2] = 0.0
    A[7, 3, 5] = np.inf
    A[8, ni + 1, 2] = np.nan
    smap = gh.StaticCondensationMap([1], [2], ctx)

    def run(cells):
        with ctx.stream():
            at = torch.as_tensor(cells, device="cuda")
            Ad = torch.as_tensor(A, device="cuda")[at]
            bd = torch.as_tensor(b, device="cuda")[at]
        S, g, info = smap.evaluate(Ad, bd, [ni, nb], return_info=True)
        ctx.synchronize()
        return S, g, info

    S1, g1, i1 = run(np.arange(nd))
    assert int(i1[6]) == ni // 2 + 1 and not np.any(i1[:6].cpu().numpy())
    cells = rng.integers(0, 6, nc)                  # good cells after ...
    cells[:1000] = rng.integers(0, nd, 1000)        # ... a first pass with all of them
    S, g, info = run(cells)
    at = torch.as_tensor(cells, device="cuda")
    assert torch.equal(info, i1[at])
    for got, one in ((S, S1), (g, g1)):
        assert torch.equal(torch.nan_to_num(got, 7.0), torch.nan_to_num(one[at], 7.0))
        assert torch.equal(torch.isnan(got), torch.isnan(one[at]))
