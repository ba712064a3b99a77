"""A multigrid PCG past its end: the first batch queues 8 iterations and more are taken in twos, so most of the queued
launches of a loose solve (703 workgroups) find it over, some of their waves before the workgroup that says so has
run. The iterate, the iteration count and the residual are those of the iteration that met the tolerance, bit for bit
the same from captured graphs and from single launches, in every pass.

The recursive residual is the true one to the rounding of a few products: |A| |x| 2^-49 beside it."""
import numpy as np
import pytest

from optcuts_amd import capi
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tol", [0.5, 1e-2, 1e-4])
def test_launches_past_the_end_change_nothing(tol):
    V, F, UV = height_field_disc(300, seed=4)
    n = len(V)
    e = np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]])
    e = np.unique(np.concatenate([e, e[:, ::-1]]), axis=0)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(e[:, 0], minlength=n))]).astype(np.int32)
    c = capi.Context(0)
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        I, J, vals = c.hessian_triplets()
        c.solver_set_pattern(n, ptr, e[:, 1].astype(np.int32), fixed=(0,))
        c.solver_update_a(I, J, vals)
        c.solver_set_params(capi.PRECOND_AMG, rel_tol=tol, max_iter=100)
        c.solver_set_coords(UV)
        c.solver_factorize()
        b = np.random.default_rng(0).normal(size=2 * n)
        b[:2] = 0.0
        out = []
        for k in range(8):
            c.pcg_graphs(k % 2 == 0)
            out.append((c.solver_solve(b), c.solver_last_stats()))
        x, (it, rr) = out[0]
        print("tol", tol, "iterations", it, "residual", rr, flush=True)
        assert 0 < it < 100 and rr <= tol
        for y, stats in out[1:]:
            assert stats == (it, rr) and np.array_equal(y, x)
        r = np.linalg.norm(c.solver_multiply(x) - b) / np.linalg.norm(b)
        amax = np.abs(vals).max() * 6 * 14  # a row: at most 7 blocks, each of at most 6 triangles' terms
        assert abs(r - rr) <= 2.0**-49 * amax * np.linalg.norm(x) / np.linalg.norm(b) + 1e-12
    finally:
        c.close()
