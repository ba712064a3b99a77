"""Refined Newton solves (PCG on the FP32-rounded matrix) of systems that run in one workgroup: 1,024 rows, the limit of
one row a thread, and 2,025, two a thread, whose second rows come from the FP32 slot-major copy. The same statement as
the 5k-face test's: the FP64 residual reaches 1e-12 in two or more passes and the energies follow the oracle's LDL^T
steps to 1e-9."""
import pytest

from oracle import oracle as O
from optcuts_amd import capi
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [32, 45])
def test_refined_jacobi_follows_the_oracle(m):
    V, F, UV = height_field_disc(m, seed=0)
    rel = 1e-16 * len(V) / (len(V) - 1)
    tr, _, _ = O.newton_run(V, F, UV, a0=1.0, max_iter=6, rel_gl2_tol=rel, allow_edec_rel_tol=False)
    c = capi.Context(0)
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        c.set_refinement(10)
        c.newton_init(a0=1.0, rel_gl2_tol=rel, allow_edec_rel_tol=False, precond=capi.PRECOND_JACOBI, pcg_rel_tol=1e-12,
                      pcg_max_iter=100000)
        passes = []
        for k in range(1, len(tr)):
            s, done = c.newton_step()
            print(k, s["E_total"], tr[k, 0], "pcg", s["pcg_iters"], "passes", s["ir_passes"], "res", s["pcg_rel_res"],
                  flush=True)
            assert s["pcg_fallback"] == 0 and s["pcg_rel_res"] <= 1e-12
            assert s["E_total"] == pytest.approx(tr[k, 0], rel=1e-9), k
            passes.append(s["ir_passes"])
            if done:
                break
        assert max(passes) >= 2
    finally:
        c.close()
