"""The compact layout of uploaded node arrays (the relayout of a whole-array
upload): trees that end in the one-block levels, in the first run of levels
and after it, wide and narrow levels, and arrays that are no tree. Frames on
the compact layout equal those on the direct layout bit for bit."""
import numpy as np
import pytest

import qubatron_amd as q

pytestmark = pytest.mark.gpu
BC = np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32)


def _frames(ctx, nodes, levels):
    ctx.upload_octree(nodes)
    ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    n = 4096
    ctx.upload_model(np.full((n, 3), 0.5, np.float32), np.full((n, 3), 0.57735, np.float32))
    v = q.view((880.0, 820.0, 960.0), (0.3, 0.1), 128, 96, BC, levels)
    light = np.array([[910.5, 990.25, 870.0]], np.float32)
    out = []
    for layout in (0, 1):
        ctx.set_tuning(layout=layout)
        ctx.render(v, light, q.OUT_ALL)
        f = ctx.read_frame(0)
        out.append((f, ctx.stats()["compact"]))
    ctx.set_tuning(layout=0)
    return out


@pytest.mark.parametrize("levels", [1, 2, 4, 5, 6, 11, 12, 13, 14, 21, 24])
@pytest.mark.parametrize("n", [1, 300, 40000])
def test_relayout_levels(gpu_ctx, levels, n):
    rng = np.random.default_rng(levels * 7 + n)
    pts = rng.uniform(0.5, 1799.5, (n, 3)).astype(np.float32)
    if levels > 14:
        pts = pts[:300]
    print(f"[case] {len(pts)} points, {levels} levels", flush=True)
    nodes = q.octree_from_points(pts, BC, levels).nodes()
    (a, ca), (b, cb) = _frames(gpu_ctx, nodes, levels)
    assert ca == 1 and cb == 0
    assert gpu_ctx.layout_stats()[2] == nodes.shape[0]
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k


@pytest.mark.parametrize("levels,parent_depth", [(6, 1), (6, 4), (9, 8), (13, 12)])
def test_relayout_refuses_shared_children(gpu_ctx, levels, parent_depth):
    """A slot that points at a node another slot holds already: not a tree, the direct layout is used."""
    rng = np.random.default_rng(levels)
    nodes = q.octree_from_points(rng.uniform(0.5, 1799.5, (60, 3)).astype(np.float32), BC, levels).nodes()
    level = np.zeros(nodes.shape[0], np.int64)
    for i in range(nodes.shape[0]):  # parents come before their children
        level[nodes[i, :8][nodes[i, :8] > 0]] = level[i] + 1
    at = np.flatnonzero(level == parent_depth)
    two = [i for i in at if (nodes[i, :8] > 0).sum() < 8][:2]
    src = nodes[two[0], :8].max()
    free = int(np.flatnonzero(nodes[two[1], :8] == 0)[0])
    nodes = nodes.copy()
    nodes[two[1], free] = src
    print(f"[case] shared child at depth {parent_depth + 1} of {levels}", flush=True)
    (a, ca), (b, cb) = _frames(gpu_ctx, nodes, levels)
    assert ca == 0 and cb == 0
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k
