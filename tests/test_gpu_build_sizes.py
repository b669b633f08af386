"""The GPU builder at the sizes where its passes can go wrong: around the
sorted positions a wave handles (1024) and a block (4096), a depth with few
and with many nodes, 32-bit and 64-bit keys, one level, heavy duplicates. The
node array equals the host builder's, and a frame of the built tree (its
compact layout, written by the builder) equals one of the uploaded array."""
import numpy as np
import pytest

import qubatron_amd as q

pytestmark = pytest.mark.gpu
BC = np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32)


def _points(n, kind, rng):
    if kind == "uniform":
        return rng.uniform(0.5, 1799.5, (n, 3)).astype(np.float32)
    if kind == "duplicates":  # a few cells hold nearly all points
        c = rng.uniform(0.5, 1799.5, (7, 3))
        return c[rng.integers(0, 7, n)].astype(np.float32)
    return (np.array([900.0, 300.0, 900.0]) + rng.normal(size=(n, 3)) * 4.0).astype(np.float32)


@pytest.mark.parametrize("levels", [1, 2, 10, 11, 12])
@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 4096, 4097, 70001])
@pytest.mark.parametrize("kind", ["uniform", "duplicates", "cluster"])
def test_build_sizes(gpu_ctx, kind, n, levels):
    rng = np.random.default_rng(n * 31 + levels)
    pts = _points(n, kind, rng)
    print(f"[case] {kind} n={n} levels={levels}", flush=True)
    gpu_ctx.upload_points(pts)
    m = gpu_ctx.build_octree(BC, levels, n)
    g = gpu_ctx.download_octree(m)
    h = q.octree_from_points(pts, BC, levels).nodes()
    assert np.array_equal(g, h)
    if n < 1023:
        return
    col, nrm = np.full((n, 3), 0.5, np.float32), np.full((n, 3), 0.57735, np.float32)
    gpu_ctx.upload_model(col, nrm)
    gpu_ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    v = q.view((880.0, 320.0, 960.0), (0.3, 0.1), 96, 64, BC, levels)
    light = np.array([[910.5, 990.25, 870.0]], np.float32)
    gpu_ctx.render(v, light, q.OUT_ALL)
    a = gpu_ctx.read_frame(0)
    assert gpu_ctx.stats()["compact"] == 1
    gpu_ctx.upload_octree(h)  # a relayout of the array
    gpu_ctx.render(v, light, q.OUT_ALL)
    b = gpu_ctx.read_frame(0)
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k
