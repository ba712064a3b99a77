"""Jacobi-PCG of small systems (one workgroup; 1,024 rows a pass, 8 blocks of a row kept, up to 2,048 rows) at its
edges: fewer rows than a wave, one row short of, at and past each pass and the limit, with a row of 40 blocks in the
first and in the last pass. A chain with random SPD couplings: eigenvalues at least d = 0.05 (the
diagonal excess) and at most 2 x 42 x 1.5 + d (twice a hub's sum of couplings), so a residual of 1e-13 leaves at most
2,530 x 1e-13 of the solution: 3e-10 against a direct solve. The plain
chain (d = 0) held at one end needs as many iterations as it has vertices, across the launches' 1,024-iteration spans;
checked there by the residual.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

from optcuts_amd import capi

pytestmark = pytest.mark.gpu


def _system(n, excess, seed):
    """Graph: the chain, and (excess > 0, n > 100) vertices 7 and n - 2 joined to 40 others. Couplings -c R R^T, c in [0.5, 1.5],
    with the rows' sums of c (times I >= R R^T) on the diagonal, which keeps it positive definite."""
    rng = np.random.default_rng(seed)
    e = {(i, i + 1) for i in range(n - 1)}
    if excess and n > 100:
        for hub in (7, n - 2):
            e |= {(min(hub, v), max(hub, v)) for v in rng.choice(n, 40, replace=False).tolist() if abs(v - hub) > 1}
    e = np.array(sorted(e))
    a = rng.uniform(0, np.pi, len(e))
    c = rng.uniform(0.5, 1.5, len(e)) if excess else np.ones(len(e))
    dirs = np.stack([np.cos(a), np.sin(a)], 1)
    B = np.einsum("e,ei,ej->eij", c, dirs, dirs) if excess else np.broadcast_to(np.eye(2), (len(e), 2, 2))
    D = np.zeros((n, 2, 2))
    for k in (0, 1):
        np.add.at(D, e[:, k], c[:, None, None] * np.eye(2))
    D += excess * np.eye(2)
    D[0] = np.eye(2)  # the fixed vertex
    I, J, V = [], [], []
    for (u, w), b in zip(e, B):
        if u == 0:
            continue
        for i in (0, 1):
            for j in (0, 1):
                I.append(2 * u + i), J.append(2 * w + j), V.append(-b[i, j])
    for v in range(n):
        for i in (0, 1):
            I.append(2 * v + i), J.append(2 * v + i), V.append(D[v, i, i])
    nb = [[] for _ in range(n)]
    for u, w in e.tolist():
        nb[u].append(w)
        nb[w].append(u)
    ptr = np.concatenate([[0], np.cumsum([len(q) for q in nb])]).astype(np.int32)
    nbr = np.array([w for q in nb for w in sorted(q)], np.int32)
    U = sp.coo_matrix((V, (I, J)), shape=(2 * n, 2 * n)).tocsr()
    return ptr, nbr, np.array(I), np.array(J), np.array(V), (U + U.T - sp.diags(U.diagonal())).tocsc(), rng


@pytest.mark.parametrize("n,excess", [(3, 0.05), (1023, 0.05), (1024, 0.05), (1025, 0.05), (2048, 0.05), (2049, 0.05),
                                      (2048, 0.0)])
def test_small_system_solves(n, excess):
    ptr, nbr, I, J, V, A, rng = _system(n, excess, n)
    b = rng.normal(size=2 * n)
    c = capi.Context(0)
    try:
        c.solver_set_pattern(n, ptr, nbr, fixed=(0,))
        c.solver_update_a(I, J, V)
        tol = 1e-13 if excess else 1e-9
        c.solver_set_params(capi.PRECOND_JACOBI, rel_tol=tol, max_iter=100000)
        c.solver_factorize()
        x = c.solver_solve(b)
        it, rr = c.solver_last_stats()
        assert rr <= tol
        if excess:
            ref = spl.spsolve(A, b)
            assert np.linalg.norm(x - ref) <= 3e-10 * np.linalg.norm(ref)
        else:
            assert it > 1024
            assert np.linalg.norm(A @ x - b) <= 1e-7 * np.linalg.norm(b)  # drift of the recursive residual
        # the cap: not converged, after exactly that many iterations
        c.solver_set_params(capi.PRECOND_JACOBI, rel_tol=1e-13, max_iter=3)
        c.solver_factorize()
        c.solver_solve(b, allow_not_converged=True)
        assert c.solver_last_stats()[0] == min(3, it)
    finally:
        c.close()
