"""The network's head and encoder weight gradients at the edges of their tiles (64 edges or vertices per tile, one
tile per workgroup up to 512): fewer rows than a tile (2x2 grid), exactly one tile of vertices (8x8), and more edge
tiles than workgroups (77x77: 35,000 edges). Checked against the float64 oracle with the GPU's bf16 operand rounding;
2e-3 of a tensor's norm as in test_gpu_gnn.py (FP32 sums against float64, ReLU and bf16 decisions within FP32
rounding of their boundary)."""
import numpy as np
import pytest

from _helpers import block_system, distort
from optcuts_amd import capi
from optcuts_amd.meshgen import height_field_disc
from oracle import gnn_oracle as G
from test_gpu_gnn import _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 8, 77])
def test_weight_gradients_at_tile_edges(m):
    V, F, UV = height_field_disc(m, 1)
    rp, ci, va, fm = block_system(V, F, distort(UV, 2, 0.1))
    th = _params(8)
    g = G.Graph(rp, ci, va, fm)
    _, ref = G.loss_and_grad(th.astype(np.float64), g, G.probes(g.nV, 2, 7), bf=True)
    net = capi.Gnn(0)
    try:
        net.set_params(th)
        net.set_system(rp, ci, va, fm)
        net.zero_grad()
        net.loss_grad(2, 7)
        got, ref = G.unflatten(net.get_grads().astype(np.float64)), G.unflatten(ref)
    finally:
        net.close()
    total = np.sqrt(sum((r ** 2).sum() for r in ref.values()))
    for name, _ in G.LAYOUT:
        err = np.linalg.norm(got[name] - ref[name])
        assert err <= 2e-3 * np.linalg.norm(ref[name]) + 1e-7 * total, (m, name, err)
