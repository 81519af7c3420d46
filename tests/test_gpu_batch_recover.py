"""Recovery of a batch's members: a class's meshes are condensed in one launch, so
what that launch keeps for the recovery has to serve every member, whatever
kernel its own number of cells takes.  Darcy classes of one row tile (2D k=3, 3D
k=1) with members on both sides of the recovery's 2,048 cells (2D with more tiles:
1,024), and members below it whose class is above, against each mesh alone and the direct solve of the
cells' interior systems; the factor slots are filled with NaN before the launch
that counts."""
import numpy as np
import pytest

from test_gpu_parity import _device_cell_systems, rel

pytestmark = pytest.mark.gpu

# (D, k, members)
CLASSES = [(2, 3, ((60, 60), (8, 8))), (2, 3, ((39, 41), (33, 31))),
           (3, 1, ((13, 13, 13), (3, 3, 3))), (3, 1, ((3, 3, 3), (12, 12, 11), (9, 9, 9))),
           (2, 4, ((33, 32), (9, 7))), (2, 5, ((6, 5), (32, 33)))]


class _Slots:
    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "version": 2,
                                         "data": (ptr, False)}


def _poison(op):
    """NaN over the mesh's factor slots (they are written by every condensation)."""
    import ctypes as C

    import torch
    from gridaphybrid import _lib
    U = C.c_void_p()
    _lib.check(_lib.lib().hdg_local_factors(op.mesh, C.byref(U), None), op.ctx.h, "factors")
    n = int(op.factor_layout().u_stride) * op.info.ncells
    op.ctx.synchronize()
    torch.as_tensor(_Slots(U.value, n), device="cuda").fill_(float("nan"))
    torch.cuda.synchronize()


def _build(ctx, D, k, cells, seed, assemble):
    import gridaphybrid as gh
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, cells)
    X = gh.HDGSpaces.darcy_baseline(model, k)
    kappa = np.random.default_rng(seed).uniform(0.5, 2.0, int(np.prod(cells)))
    return gh.HybridAffineFEOperator(gh.DarcyHDG(tau=1.0, kappa=kappa, source=3), X, X, [1, 2],
                                     [3], ctx=ctx, assemble=assemble)


@pytest.mark.parametrize("autotune", [False, True])
@pytest.mark.parametrize("D,k,members", CLASSES)
def test_members_on_both_sides_of_the_recovery_switch(ctx, D, k, members, autotune):
    import gridaphybrid as gh
    import torch
    print(f"batch recovery D={D} k={k} members={members} autotune={autotune}", flush=True)
    lams, alone = [], []
    for s, cells in enumerate(members):
        op = _build(ctx, D, k, cells, s, True)
        lams.append(np.random.default_rng(100 + s).standard_normal(op.info.nfree))
        alone.append(op.recover(lams[-1]).cpu().numpy())
        op.close()
    ops = [_build(ctx, D, k, cells, s, False) for s, cells in enumerate(members)]
    batch = gh.HybridOperatorBatch(ops, autotune=autotune)
    batch.assemble()
    for op in ops:
        _poison(op)
    batch.assemble()
    dev = [torch.as_tensor(v, device="cuda") for v in lams]
    outs = [torch.empty(op.info.nfree_total, dtype=torch.float64, device="cuda") for op in ops]
    torch.cuda.synchronize()
    batch.recover(dev, outs)
    ctx.synchronize()
    for op, lam, out, ref in zip(ops, lams, outs, alone):
        got = out.cpu().numpy()
        if autotune:
            assert rel(got, ref) < 1e-11
        else:  # the class's default family, the member's own recovery kernel
            assert np.array_equal(got, ref)
        nc, na, ni = op.info.ncells, op.info.n_flux, op.info.ni
        cnt = min(nc, 40)
        A, b = _device_cell_systems(op, 0, cnt)
        cd = np.asarray(op.cell_blocks()[2]).reshape(nc, -1)[:cnt]
        ld = np.where(cd >= 0, lam[np.maximum(cd, 0)], 0.0)
        c = b[:, :ni] - np.einsum("cij,cj->ci", A[:, :ni, ni:], ld)
        x = np.linalg.solve(A[:, :ni, :ni], c[..., None])[..., 0]
        xi = np.concatenate([got[:nc * na].reshape(nc, na)[:cnt],
                             got[nc * na:nc * ni].reshape(nc, ni - na)[:cnt]], 1)
        assert rel(xi, x) < 1e-11
    batch.close()
    for op in ops:
        op.close()
