"""The joint mode's PCG graphs across air re-meshes that keep the multigrid structure: such a step names the same
buffers as the one before (the matrix mapped onto the kept pattern stays where it is; only a Newton matrix that outgrows
its buffer moves), so its graphs are replayed and not captured anew."""
import pytest

from optcuts_amd import capi
from optcuts_amd import scaffold as air
from optcuts_amd.meshgen import height_field_disc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [capi.PRECISION_FP64, capi.PRECISION_MIXED])
def test_kept_structure_keeps_its_graphs(precision):
    m = 60
    V, F, UV = height_field_disc(m, seed=3)
    UV = UV * [1.0, 0.6]  # a map whose boundary moves for many steps
    edge = (2.0 + 2.0**0.5) / (3.0 * (m - 1))
    c = capi.Context(0)
    try:
        c.set_mesh(V, F, fixed=(0,))
        c.set_uv(UV)
        c.set_air_mesh(*air.initial_air_mesh(UV, F, edge), air.area_threshold(edge), 1e-5)
        c.newton_init(a0=1e-3, rel_gl2_tol=1e-12, allow_edec_rel_tol=False, precond=capi.PRECOND_AMG, pcg_rel_tol=1e-3,
                      pcg_max_iter=100, precision=precision)
        steps, builds = [], 0
        for _ in range(12):
            kept = c.setup_times()["amg_kept_remeshes"]
            s, _ = c.newton_step()
            steps.append((kept, c.pcg_graph_builds() - builds, s["pcg_iters"], s["pcg_fallback"]))
            builds = c.pcg_graph_builds()
            steps[-1] += (c.scaffold_update(mode=capi.SCAFFOLD_REMESH)[1],)
        for k, row in enumerate(steps):
            print(k, "kept re-meshes %d, graphs %d, iterations %d, fallback %d, then flips %d" % row, flush=True)
        # a step after a flip that is at least the second re-mesh on its structure
        again = [b for (kept, b, *_), (*_, flips) in zip(steps[1:], steps) if flips > 0 and kept >= 2]
        assert len(again) >= 2
        assert 0 in again
    finally:
        c.close()
