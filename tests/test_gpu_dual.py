"""Both trees on their compact layouts: frames equal those on the direct
layout bit for bit, before and after child slots of both trees are zeroed in
place (the compact child blocks then have slots without a child)."""
import numpy as np
import pytest

import qubatron_amd as q

pytestmark = pytest.mark.gpu


def _equal(ctx, bc, levels, what):
    lo = np.array([bc[0], bc[1] - bc[3], bc[2] - bc[3]])
    at = (lo + np.array([0.49, 0.45, 0.53]) * bc[3]).astype(np.float32)
    v = q.view(at, (0.3, 0.1), 160, 120, bc, levels)
    lights = (lo + np.array([[0.506, 0.55, 0.483], [0.3, 0.8, 0.6]]) * bc[3]).astype(np.float32)
    for mask in (q.OUT_ALL, q.OUT_ALL | q.RENDER_COUNT):
        out = []
        for layout in (0, 1):
            ctx.set_tuning(layout=layout)
            ctx.render(v, lights, mask)
            out.append(ctx.read_frame(0))
            st = ctx.stats()
            assert st["dual"] == 1 and st["compact"] == 1 - layout, what
        ctx.set_tuning(layout=0)
        for k in out[0]:
            assert np.array_equal(out[0][k].view(np.uint8), out[1][k].view(np.uint8)), (what, mask, k)


@pytest.mark.parametrize("bc", [(0.0, 1800.0, 1800.0, 1800.0), (0.3, 1000.7, 1001.1, 1000.7)])
@pytest.mark.parametrize("levels,n,ndyn", [(1, 5, 3), (2, 60, 40), (7, 3000, 500), (7, 500, 20000), (12, 20000, 20000)])
def test_dual_layouts_agree(gpu_ctx, bc, levels, n, ndyn):
    rng = np.random.default_rng(levels * 100 + ndyn)
    lo = np.array([bc[0], bc[1] - bc[3], bc[2] - bc[3]])
    bc = np.array(bc, np.float32)
    trees = []
    for t, k in enumerate((n, ndyn)):
        pts = (lo + rng.uniform(0.001, 0.999, (k, 3)) ** (1 + t) * bc[3]).astype(np.float32)
        nodes = q.octree_from_points(pts, bc, levels).nodes()
        gpu_ctx.upload_octree(nodes, dynamic=t == 1)
        gpu_ctx.upload_model(rng.uniform(0, 1, (k, 3)).astype(np.float32),
                             np.full((k, 3), 0.57735, np.float32), dynamic=t == 1)
        trees.append(nodes.copy())
    print(f"[case] dual {levels} levels, {n} + {ndyn} points", flush=True)
    _equal(gpu_ctx, bc, levels, "as uploaded")
    for t, nodes in enumerate(trees):
        nz = np.argwhere(nodes[:, :8] > 0)
        for i, o in nz[rng.permutation(len(nz))[:min(60, len(nz) // 2)]]:
            nodes[i, o] = 0
            gpu_ctx.upload_octree(nodes, dynamic=t == 1, start_node=int(i), end_node=int(i) + 1)
    _equal(gpu_ctx, bc, levels, "slots zeroed")
