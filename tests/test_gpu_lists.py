"""The list of shaded pixels at the sizes where its launches change shape
(one block, a last block without items, offsets summed by every block and
offsets from a scan): frames equal those of the merged launch, which makes no
list, bit for bit."""
import numpy as np
import pytest

import qubatron_amd as q

pytestmark = pytest.mark.gpu
BC = np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32)


@pytest.mark.parametrize("w,h", [(1, 1), (64, 32), (64, 33), (2048, 2040), (2048, 2047), (2120, 2048)])
def test_frames_with_and_without_a_list(gpu_ctx, w, h):
    rng = np.random.default_rng(w + h)
    pts = rng.uniform(300.0, 1500.0, (3000, 3)).astype(np.float32)
    gpu_ctx.upload_octree(q.octree_from_points(pts, BC, 7).nodes())
    gpu_ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    gpu_ctx.upload_model(rng.uniform(0, 1, (3000, 3)).astype(np.float32), np.full((3000, 3), 0.57735, np.float32))
    v = q.view((900.0, 900.0, 1790.0), (0.1, 0.05), w, h, BC, 7)
    lights = np.array([[910.5, 990.25, 1700.0], [300.0, 1500.0, 1200.0]], np.float32)
    print(f"[case] {w} x {h}", flush=True)
    out = []
    for merge in (0, 2):
        gpu_ctx.set_tuning(merge=merge)
        gpu_ctx.render(v, lights, q.OUT_ALL)
        out.append((gpu_ctx.read_frame(0), gpu_ctx.stats()["shadow_rays"]))
    gpu_ctx.set_tuning(merge=1)
    (a, na), (b, nb) = out
    assert w * h < 1000 or na > 0
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k
