"""The path of long loosely stopped solves is fixed by the order and the rounding of their sums: a Newton step of the
learned form (PCG to 5e-3 over some hundred iterations) stops at another iterate once one sum is formed differently, by
up to a few percent of the map. These iteration counts and residuals were recorded with the plain form of the kernels
(one load after another), so a kernel that adds the same terms in another order shows here; whoever changes the order
on purpose records them anew.
Residuals to 1e-9: a solve on the same path differs by roundings of the last sum, one on another path by 1e-3. Block
IC(0) and Jacobi solves beside them on either side of the size where the PCG product's workgroups change."""
import numpy as np
import pytest

from optcuts_amd import capi, learned
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,seed,precond,tol,iters,rel_res", [
    (30, 1, capi.PRECOND_LEARNED, 5e-3, 35, 0.0048552352927754535),
    (100, 3, capi.PRECOND_LEARNED, 5e-3, 167, 0.00497586909217714),
    (159, 3, capi.PRECOND_LEARNED, 5e-3, 444, 0.0049625514338662345),
    (159, 42, capi.PRECOND_LEARNED, 5e-3, 235, 0.0048858437616129263),
    (159, 80, capi.PRECOND_LEARNED, 5e-3, 454, 0.0049005555350356391),
    (163, 215466, capi.PRECOND_LEARNED, 5e-3, 422, 0.0047684948825329199),
    (317, 2, capi.PRECOND_LEARNED, 5e-3, 525, 0.0049382627616300009),
    (100, 1, capi.PRECOND_IC0, 5e-3, 197, 0.0046296395091234947),
    (100, 1, capi.PRECOND_JACOBI, 1e-10, 1882, 9.6055559367024656e-11),
    (317, 1, capi.PRECOND_JACOBI, 1e-10, 5522, 9.702887976954107e-11),
    (400, 2, capi.PRECOND_JACOBI, 1e-10, 7027, 9.7623780559809568e-11),
])
def test_step_takes_its_recorded_path(m, seed, precond, tol, iters, rel_res):
    V, F, UV = height_field_disc(m, seed=seed)
    c, net = capi.Context(0), None
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        if precond == capi.PRECOND_LEARNED:
            net = capi.Gnn(0)
            net.set_params(np.load(learned.DEFAULT_WEIGHTS))
            c.set_learned(net)
        c.newton_init(a0=1.0, rel_gl2_tol=1e-30, allow_edec_rel_tol=False, precond=precond, pcg_rel_tol=tol,
                      pcg_max_iter=200000,
                      precision=capi.PRECISION_MIXED if precond == capi.PRECOND_LEARNED else capi.PRECISION_FP64)
        s, _ = c.newton_step()
        print(m, seed, precond, s["pcg_iters"], repr(s["pcg_rel_res"]), flush=True)
        assert s["pcg_iters"] == iters
        assert s["pcg_rel_res"] == pytest.approx(rel_res, rel=1e-9)
    finally:
        c.close()
        if net is not None:
            net.close()
