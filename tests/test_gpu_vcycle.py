"""One multigrid Newton step at the sizes where its kernels change: 9 vertices, 144 (the lambda_max estimate of a whole
level in one launch; levels of at most 128 nodes), 2,025, and on both sides of 131,072 rows (coarse correction and
first post-smoothing step in one launch below) and of 1,024 workgroups of 256 triangles in the line search (131,044
vertices and 260,642 faces, 132,496 and 263,538).

- The step's direction solves its own exported system. The direction is (UV1 - UV0) / step: rounding of the positions
  (2^-53 each) leaves |A|_inf 2^-52 max|UV| sqrt(2 n) / step in the residual, beside the PCG tolerance times |b|
  (recursive residual: twice that is allowed). A wrong level would not reach the tolerance in 120 iterations.
- The line search's energy of the accepted positions is the energy kernel's: both add the same FP64 terms in
  compensated sums, each term within a few hundred roundings, 1e-13 relative.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from optcuts_amd import capi
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [3, 12, 45, 362, 364])
def test_multigrid_newton_step(m):
    V, F, UV = height_field_disc(m, seed=1)
    n, tol = len(V), 1e-9
    c = capi.Context(0)
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        c.newton_init(a0=1.0, rel_gl2_tol=1e-16, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG,
                      pcg_rel_tol=tol, pcg_max_iter=120)
        E0 = c.energy()
        s, _ = c.newton_step()
        assert s["pcg_fallback"] == 0 and 0 < s["pcg_iters"] < 120
        rp, ci, va, b, _ = c.get_system()
        A = sp.bsr_matrix((va.reshape(-1, 2, 2), ci, rp), shape=(2 * n, 2 * n)).tocsr()
        UV1 = c.get_uv()
        d = (UV1 - UV).ravel() / s["step"]
        slack = abs(A).sum(1).max() * 2.0**-52 * np.abs(UV1).max() * np.sqrt(2 * n) / s["step"]
        r = np.linalg.norm(A @ d - b.ravel())
        print("m", m, "pcg", s["pcg_iters"], "residual", r, "of", np.linalg.norm(b), "slack", slack, flush=True)
        assert r <= 2 * tol * np.linalg.norm(b) + slack
        E1 = c.energy()
        assert E1 < E0 and abs(s["E_SD"] - E1) <= 1e-13 * E1
    finally:
        c.close()
