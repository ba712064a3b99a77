"""Jacobi-PCG of small systems with long rows: the one-workgroup form gives a row to one thread and every row to one
CU, so patterns past its limits (a row of 64 blocks, 4,096 blocks past the eighth of their rows, shared where both
occur) take the two launches an iteration that larger systems take.

Scalar couplings c in [0.5, 1.5] on both coordinates plus d = 0.05 on the diagonal: eigenvalues from d to at most twice
the longest row's couplings, 2 x 1.5 x longest + d, so a residual of 1e-13 leaves 1e-13 x that / d of the solution."""
import time

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

from optcuts_amd import capi

pytestmark = pytest.mark.gpu


def _system(n, hubs, length, band, seed):
    rng = np.random.default_rng(seed)
    e = {(i, i + k) for k in range(1, band + 1) for i in range(n - k)}
    for h in hubs:
        e |= {(min(h, v), max(h, v)) for v in rng.choice(n, length, replace=False).tolist() if v != h}
    e = np.array(sorted(e))
    c = rng.uniform(0.5, 1.5, len(e))
    D = np.full(n, 0.05)
    np.add.at(D, e[:, 0], c)
    np.add.at(D, e[:, 1], c)
    D[0] = 1.0
    f = e[:, 0] != 0
    I = np.concatenate([2 * e[f, 0] + k for k in (0, 1)] + [np.arange(2 * n)])
    J = np.concatenate([2 * e[f, 1] + k for k in (0, 1)] + [np.arange(2 * n)])
    V = np.concatenate([-c[f], -c[f], np.repeat(D, 2)])
    d = np.concatenate([e, e[:, ::-1]])
    d = d[np.lexsort((d[:, 1], d[:, 0]))]
    ptr = np.concatenate([[0], np.cumsum(np.bincount(d[:, 0], minlength=n))]).astype(np.int32)
    U = sp.coo_matrix((V, (I, J)), shape=(2 * n, 2 * n)).tocsr()
    return ptr, d[:, 1].astype(np.int32), I, J, V, (U + U.T - sp.diags(U.diagonal())).tocsc(), rng


def _context(n, ptr, nbr, I, J, V, tol, max_iter):
    c = capi.Context(0)
    c.solver_set_pattern(n, ptr, nbr, fixed=(0,))
    c.solver_update_a(I, J, V)
    c.solver_set_params(capi.PRECOND_JACOBI, rel_tol=tol, max_iter=max_iter)
    c.solver_factorize()
    return c


# one hub of about 60 and of about 73 blocks (either side of the limit for one row), three of 43, one of all vertices;
# bands of 9 and of 13 blocks a row (either side of the limit for all rows)
@pytest.mark.parametrize("n,hubs,length,band", [(1024, [500], 57, 1), (2048, [2046], 70, 1), (2048, [7, 1500, 2046], 40, 1),
                                                (1500, [3], 1499, 1), (2048, [], 0, 4), (2048, [], 0, 6)])
def test_long_rows_solve(n, hubs, length, band):
    ptr, nbr, I, J, V, A, rng = _system(n, hubs, length, band, n + length)
    b = rng.normal(size=2 * n)
    c = _context(n, ptr, nbr, I, J, V, 1e-13, 100000)
    try:
        x = c.solver_solve(b)
    finally:
        c.close()
    longest = np.diff(ptr).max() + 1
    ref = spl.spsolve(A, b)
    assert np.linalg.norm(x - ref) <= 1e-13 * (3 * longest + 0.05) / 0.05 * np.linalg.norm(ref)


def test_long_rows_are_not_walked_by_one_workgroup():
    """65 blocks in every row: 2,048 rows, which may take one workgroup, cost an iteration what 2,049 do, which may not
    (254 and 12 us where the row count alone decided; a factor of 3 is allowed for)."""
    per_iteration = []
    for n in (2048, 2049):
        ptr, nbr, I, J, V, A, rng = _system(n, [], 0, 32, n)
        b = rng.normal(size=2 * n)
        c = _context(n, ptr, nbr, I, J, V, 1e-150, 80)
        try:
            c.solver_solve(b, allow_not_converged=True)
            best = 1e9
            for _ in range(10):
                t = time.perf_counter()
                c.solver_solve(b, allow_not_converged=True)
                best = min(best, time.perf_counter() - t)
            assert c.solver_last_stats()[0] == 80
            per_iteration.append(best / 80)
        finally:
            c.close()
    print("seconds an iteration", per_iteration, flush=True)
    assert per_iteration[0] < 3 * per_iteration[1]
