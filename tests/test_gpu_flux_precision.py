"""Elasticity's reduced systems in the orthonormal basis of the displacement.

S is no further from the Schur complement of the weak form, integrated and
eliminated in extended precision, than the dense FP64 elimination of all the
cell's rows (64 units of rounding of the largest entry where both are below
that).  S does not depend on the interior bases, so the reference takes products
of Legendre polynomials; only its trace functions are the nodal ones.

The factors of hdg_local_factors are those of the displacement's own basis and
stay current for whoever has asked once: after a further condensation of the
mesh, and after a batch's."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_batch_recover import _Slots, _poison
from test_gpu_parity import _device_cell_systems, check_local_factors

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _operator(ctx, D, k, n, seed=3, family=None, projection=False, assemble=True):
    import gridaphybrid as gh
    model = gh.CartesianDiscreteModel((0.0, 1.0) * D, (n,) * D)
    X = gh.HDGSpaces.elasticity(model, k)
    nu = np.random.default_rng(seed).uniform(0.2, 0.4, n ** D)
    wf = gh.ElasticityHDG(tau=float(n), nu=nu, E=1.0, source=12,
                          bulk_to_skeleton_projection=projection)
    return gh.HybridAffineFEOperator(wf, X, X, [1, 2], [3], ctx=ctx, family=family,
                                     assemble=assemble)


def _gauss(m):
    """Gauss points and weights on [0, 1] in extended precision."""
    x, one = np.polynomial.legendre.leggauss(m)[0].astype(LD), np.ones(m, LD)
    for _ in range(4):
        p0, p1 = one, x
        for j in range(2, m + 1):
            p0, p1 = p1, ((2 * j - 1) * x * p1 - (j - 1) * p0) / j
        dp = m * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / dp
    return (x + 1) / 2, 1 / ((1 - x * x) * dp * dp)


def _legendre(k, x):
    """Orthonormal Legendre polynomials of degree 0..k on [0, 1]: values,
    derivatives, [point, degree]."""
    t = 2 * x - 1
    v, d = [np.ones_like(t), t], [np.zeros_like(t), np.ones_like(t)]
    for j in range(2, k + 1):
        v.append(((2 * j - 1) * t * v[-1] - (j - 1) * v[-2]) / j)
        d.append(d[-2] + (2 * j - 1) * v[-2])
    c = np.sqrt(2 * np.arange(k + 1, dtype=LD) + 1)
    return np.stack(v[:k + 1], 1) * c, 2 * np.stack(d[:k + 1], 1) * c


def _modes(D, k, x):
    """Products of Legendre polynomials of total degree <= k at points x [q, D]:
    values [q, n], derivatives [D, q, n]."""
    e = np.array([i for i in np.ndindex(*(k + 1,) * D) if sum(i) <= k])
    v, d = zip(*[_legendre(k, x[:, a]) for a in range(D)])
    val = np.prod([v[a][:, e[:, a]] for a in range(D)], axis=0)
    der = [np.prod([(d if a == g else v)[a][:, e[:, a]] for a in range(D)], axis=0)
           for g in range(D)]
    return val, np.stack(der)


def _trace_nodes(d, k):
    """Nodes of the trace element of order k: vertices, edges, interior."""
    if d == 1:
        return np.array([[0], [k]] + [[i] for i in range(1, k)], LD) / k
    pts = [(0, 0), (k, 0), (0, k)]
    for fixed in (1, 0):                 # edges along the first, then the second direction
        for c in (0, k):
            pts += [(i, c) if fixed else (c, i) for i in range(1, k) if i + c <= k]
    pts += [(i, j) for j in range(1, k) for i in range(1, k) if i + j <= k]
    return np.array(pts, LD) / k


def _inv(M):
    n = len(M)
    M = np.concatenate([M, np.eye(n, dtype=LD)], 1)
    for c in range(n):
        p = c + int(np.argmax(np.abs(M[c:, c])))
        M[[c, p]] = M[[p, c]]
        M[c] /= M[c, c]
        f = M[:, c].copy()
        f[c] = 0
        M -= np.outer(f, M[c])
    return M[:, n:]


def _rule(d, m):
    x, w = _gauss(m)
    i = np.array(list(np.ndindex(*(m,) * d))).reshape(-1, d)
    return x[i], np.prod(w[i], axis=1)


def _weak_form_schur(D, k, n, nu, projection):
    """S of one cell of the n^D mesh of the unit cube, tau = n, E = 1."""
    h, tau = 1 / LD(n), LD(n)
    x, w = _rule(D, k + 3)
    P, dP = _modes(D, k, x)
    Q = _modes(D, k + 1, x)[0]
    nodes = _trace_nodes(D - 1, k)
    V = _inv(_modes(D - 1, k, nodes)[0])          # nodal trace functions from modes
    pairs = [(i, j) for i in range(D) for j in range(i, D)]
    E = np.zeros((len(pairs), D, D), LD)
    for s, (i, j) in enumerate(pairs):
        E[s, i, j] = E[s, j, i] = 1
    nf, nu_, nt = P.shape[1], Q.shape[1], len(nodes)
    na, ni = len(pairs) * nf, len(pairs) * nf + D * nu_
    A = np.zeros((ni + 2 * D * D * nt,) * 2, LD)
    fl = lambda s: slice(s * nf, (s + 1) * nf)                                      # noqa: E731
    po = lambda c: slice(na + c * nu_, na + (c + 1) * nu_)                          # noqa: E731
    tr = lambda f, c: slice(ni + (f * D + c) * nt, ni + (f * D + c + 1) * nt)       # noqa: E731
    C = (1 + LD(nu)) * np.einsum("sij,rij->sr", E, E)
    C -= LD(nu) * np.outer(np.einsum("sii->s", E), np.einsum("sii->s", E))
    M = P.T @ (w[:, None] * P)
    G = [dP[j].T @ (w[:, None] * Q) for j in range(D)]
    for s in range(len(pairs)):
        for r in range(len(pairs)):
            A[fl(s), fl(r)] = C[s, r] * h ** D * M
        for c in range(D):
            A[fl(s), po(c)] = h ** (D - 1) * sum(E[s, c, j] * G[j] for j in range(D))
            A[po(c), fl(s)] = -A[fl(s), po(c)].T
    y, wf = _rule(D - 1, k + 3)
    m = _modes(D - 1, k, y)[0] @ V
    area = h ** (D - 1)
    for f in range(2 * D):
        fix = D - 1 - f // 2
        xi = np.insert(y, fix, LD(f % 2), axis=1)
        p, q = _modes(D, k, xi)[0], _modes(D, k + 1, xi)[0]
        pm, qm = p.T @ (wf[:, None] * m), q.T @ (wf[:, None] * m)
        mm, qq = m.T @ (wf[:, None] * m), q.T @ (wf[:, None] * q)
        if projection:
            qq = qm @ _inv(mm) @ qm.T
        for c in range(D):
            for s in range(len(pairs)):
                t = (E[s, c, fix] if f % 2 else -E[s, c, fix]) * area * pm
                A[fl(s), tr(f, c)] -= t
                A[tr(f, c), fl(s)] += t.T
            A[po(c), po(c)] += tau * area * qq
            A[po(c), tr(f, c)] -= tau * area * qm
            A[tr(f, c), po(c)] -= tau * area * qm.T
            A[tr(f, c), tr(f, c)] += tau * area * mm
    for c in range(ni):                           # partial pivoting
        i = c + int(np.argmax(np.abs(A[c:ni, c])))
        A[[c, i]] = A[[i, c]]
        A[c + 1:, c + 1:] -= np.outer(A[c + 1:, c] / A[c, c], A[c, c + 1:])
    return A[ni:, ni:]


@pytest.mark.parametrize("D,k,projection", [
    (2, 2, False), (2, 3, True), (3, 1, False), (3, 2, False), (3, 2, True), (3, 3, False)])
def test_schur_complement_no_further_than_dense(ctx, D, k, projection):
    print(f"flux precision D={D} k={k} projection={projection}", flush=True)
    n = 3
    ops = [_operator(ctx, D, k, n, family=8, projection=projection)]
    size = ops[0].info.ni + ops[0].info.nb
    dense = 4 if size > 300 else 5 if size > 72 else 1
    ops.append(_operator(ctx, D, k, n, family=dense, projection=projection))
    assert [op.factor_rows()[1] for op in ops] == [8, dense]
    nu = np.random.default_rng(3).uniform(0.2, 0.4, n ** D)
    err = [0.0, 0.0]
    for c in (0, 4, n ** D - 1):
        ref = _weak_form_schur(D, k, n, nu[c], projection)
        for t, op in enumerate(ops):
            d = np.abs(op.cell_blocks()[0][c] - ref).max() / np.abs(ref).max()
            err[t] = max(err[t], float(d))
    print(f"S: family 8 {err[0]:.1e} dense {err[1]:.1e}", flush=True)
    assert err[0] <= max(err[1], 64 * 2.0 ** -53)
    for op in ops:
        op.close()


def test_factors_stay_current(ctx):
    import gridaphybrid as gh
    import torch
    print("factors of the displacement's own basis", flush=True)
    op = _operator(ctx, 3, 2, 2)
    assert op.factor_rows() == (60, 8)
    A, b = _device_cell_systems(op, 0, 8)
    U, Y = op.local_factors()
    check_local_factors(op, A, b, U, Y, 8)
    ptr = C.c_void_p()
    gh._lib.check(gh._lib.lib().hdg_local_factors(op.mesh, C.byref(ptr), None), ctx.h, "factors")
    n = op.info.ncells * int(op.factor_layout().u_stride)
    at = torch.as_tensor(_Slots(ptr.value, n), device="cuda")
    _poison(op)
    op.assemble()
    ctx.synchronize()
    rows = 60 * 61 // 2
    got = at.reshape(op.info.ncells, -1)[:, :rows].cpu().numpy()
    iu = np.tril_indices(60)            # packed by columns
    assert np.array_equal(got, U.transpose(0, 2, 1)[:, iu[0], iu[1]])
    # in a batch (its slots are others: asked again after the first launch)
    mesh2 = _operator(ctx, 3, 2, 2, seed=9, assemble=False)
    batch = gh.HybridOperatorBatch([op, mesh2], autotune=False)
    batch.assemble()
    U1, Y1 = op.local_factors()
    batch.assemble()
    U2, Y2 = op.local_factors()
    for got in ((U1, Y1), (U2, Y2)):
        assert np.array_equal(got[0], U) and np.array_equal(got[1], Y)
    ref = O.hdg_solve(O.Problem.elasticity(3, 2, tau=2.0, nu=0.3, mms=O.ELAS_MMS_SIN), (2,) * 3,
                      coef=np.random.default_rng(3).uniform(0.2, 0.4, 8))
    S, g, _ = op.cell_blocks()
    assert np.max(np.abs(S - ref.S)) < 1e-12 * np.max(np.abs(ref.S))
    batch.close()
    op.close()
    mesh2.close()
