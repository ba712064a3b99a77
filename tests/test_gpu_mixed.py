"""The mixed form (FP32 element terms, FP32-stored multigrid).

- One Newton step at the sizes where the multigrid's kernels change (9, 144, 2,025, 131,044 and 132,496 vertices): the
  direction solves the exported FP64 system. It is (UV1 - UV0) / step: rounding of the positions leaves
  |A|_inf 2^-52 max|UV| sqrt(2 n) / step in the residual, beside the PCG tolerance times |b| (recursive residual: twice
  that is allowed).
- Ten joint-mode steps on a closed surface (perturbed icosphere, 100,820 faces): no fallback, at most a third more PCG
  iterations than the FP64 form, and its energy: each step's direction is off by at most the PCG tolerance, 1e-3, which
  a Newton step near the minimum turns into 1e-6 of the energy."""
import numpy as np
import pytest
import scipy.sparse as sp

from optcuts_amd import capi
from optcuts_amd import workloads as W
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [3, 12, 45, 362, 364])
def test_mixed_multigrid_newton_step(m):
    V, F, UV = height_field_disc(m, seed=1)
    n, tol = len(V), 1e-4
    c = capi.Context(0)
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        c.newton_init(a0=1.0, rel_gl2_tol=1e-16, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG,
                      pcg_rel_tol=tol, pcg_max_iter=120, precision=capi.PRECISION_MIXED)
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
        assert c.energy() < E0
    finally:
        c.close()


def test_mixed_joint_mode_needs_no_fallback():
    steps, its, energy = {}, {}, {}
    c = capi.Context(0)
    try:
        w = W.prepare_closed(c, "icosphere_100k")
        for precision in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
            W.restart(c, w)
            c.newton_init(a0=w["a0"], rel_gl2_tol=1e-12, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG,
                          pcg_rel_tol=1e-3, pcg_max_iter=100, precision=precision)
            total = 0
            for _ in range(10):
                s, _ = c.newton_step()
                c.scaffold_update()
                assert s["pcg_fallback"] == 0
                total += s["pcg_iters"]
            its[precision], energy[precision] = total, s["E_SD"]
        print("iterations", its, "energies", energy, flush=True)
        assert its[capi.PRECISION_MIXED] <= its[capi.PRECISION_FP64] * 4 / 3
        assert abs(energy[capi.PRECISION_MIXED] - energy[capi.PRECISION_FP64]) <= 1e-6 * energy[capi.PRECISION_FP64]
    finally:
        c.close()
