"""The multigrid only reads the matrix it is handed: a zero diagonal entry (a vertex that no triangle or triplet
touches) is replaced in the hierarchy and not in the matrix that PCG and oc_solver_multiply use, on hierarchies of one
level (the coarsest solve alone: a dense inverse, or diagonal blocks where every vertex is isolated) and of more.

Products: each row adds at most 5 blocks, rounded 10 times: 2^-49 of the sum of magnitudes; bitwise the same before and
after the set-up. Solutions: condition at most 2 x 8 / 0.1 (Gershgorin and the diagonal excess), so a residual of 1e-12
leaves 2e-10.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from optcuts_amd import capi
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


def _grid_laplacian(m, isolated, seed):
    """Two uncoupled 5-point Laplacians (+ 0.1 on the diagonal) on an m x m grid, vertex 0 fixed, then `isolated`
    vertices without neighbours, every second with a zero block."""
    rng = np.random.default_rng(seed)
    n = m * m + isolated
    e = [(i, i + 1) for i in range(m * m - 1) if i % m < m - 1] + [(i, i + m) for i in range(m * m - m)]
    e = np.array(e, int).reshape(-1, 2)
    c = rng.uniform(0.5, 1.0, len(e))
    diag = np.zeros(n)
    np.add.at(diag, e[:, 0], c)
    np.add.at(diag, e[:, 1], c)
    diag[:m * m] += 0.1
    diag[0] = 1.0
    diag[m * m::2] = 0.0
    diag[m * m + 1::2] = 2.0
    free = e[:, 0] != 0
    I = np.concatenate([2 * e[free, 0] + k for k in (0, 1)] + [np.arange(2 * n)])
    J = np.concatenate([2 * e[free, 1] + k for k in (0, 1)] + [np.arange(2 * n)])
    V = np.concatenate([-c[free], -c[free], np.repeat(diag, 2)])
    nb = [[] for _ in range(n)]
    for u, w in e.tolist():
        nb[u].append(w)
        nb[w].append(u)
    ptr = np.concatenate([[0], np.cumsum([len(q) for q in nb])]).astype(np.int32)
    nbr = np.array([w for q in nb for w in sorted(q)], np.int32)
    U = sp.coo_matrix((V, (I, J)), shape=(2 * n, 2 * n)).tocsr()
    return n, ptr, nbr, I, J, V, (U + U.T - sp.diags(U.diagonal())).tocsr(), diag


@pytest.mark.parametrize("m,isolated", [(3, 1), (1, 100), (20, 7)])
def test_factorize_leaves_the_matrix_as_it_was(m, isolated):
    n, ptr, nbr, I, J, V, A, diag = _grid_laplacian(m, isolated, m)
    rng = np.random.default_rng(1)
    x, b = rng.normal(size=(2, 2 * n))
    on = np.repeat(diag != 0.0, 2)
    c = capi.Context(0)
    try:
        c.solver_set_pattern(n, ptr, nbr, fixed=(0,))
        c.solver_update_a(I, J, V)
        c.solver_set_params(capi.PRECOND_AMG, rel_tol=1e-12, max_iter=200)
        c.solver_set_coords(rng.normal(size=(n, 2)))
        before = c.solver_multiply(x)
        assert np.all(np.abs(before - A @ x) <= 2.0**-49 * (abs(A) @ np.abs(x)))
        c.solver_factorize()
        assert np.array_equal(c.solver_multiply(x), before)
        # consistent: the undetermined entries stay zero
        y = c.solver_solve(np.where(on, b, 0.0))
        ref = np.zeros(2 * n)
        ref[on] = np.linalg.solve(A[on][:, on].toarray(), b[on])
        assert c.solver_last_fallback() == 0
        assert np.all(y[~on] == 0.0) and np.linalg.norm(y - ref) <= 2e-10 * np.linalg.norm(ref)
        # inconsistent: no solution is claimed
        try:
            c.solver_solve(b, allow_not_converged=True)
            assert c.solver_last_stats()[1] > 1e-12
        except capi.OCError as err:
            assert err.status == -8  # breakdown
        assert np.array_equal(c.solver_multiply(x), before)
    finally:
        c.close()


def test_newton_system_is_the_jacobi_forms():
    V, F, UV = height_field_disc(3, seed=2)
    V, UV = np.vstack([V, [[2.0, 2.0, 0.0]]]), np.vstack([UV, [[2.0, 2.0]]])  # one vertex in no triangle
    systems = []
    for precond in (capi.PRECOND_JACOBI, capi.PRECOND_AMG):
        c = capi.Context(0)
        try:
            c.set_mesh(V, F, fixed=(0,))
            c.set_uv(UV)
            c.newton_init(a0=1.0, rel_gl2_tol=1e-16, allow_edec_rel_tol=False, precond=precond, pcg_rel_tol=1e-9)
            c.newton_step()
            systems.append(c.get_system()[2].reshape(-1, 4))
        finally:
            c.close()
    assert np.array_equal(*systems)
    assert np.all(systems[0][-1] == 0.0)
