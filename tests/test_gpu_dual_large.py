"""Both trees walked where the dynamic tree has more than 2^24 nodes: the
compact layouts take part, and frames equal those on the direct layout bit for
bit."""
import numpy as np
import pytest

import qubatron_amd as q

pytestmark = pytest.mark.gpu


def test_dynamic_tree_above_2_24_nodes():
    a, b = q.Scene(2, seed=3, npoints=500000), q.Scene(2, seed=9, npoints=8000000)
    with q.Context(0) as ctx:
        for sc, dyn in ((a, False), (b, True)):
            pnt, nrm, col = sc.points()
            ctx.upload_points(pnt, dynamic=dyn)
            ctx.upload_model(col, nrm, dynamic=dyn)
            n = ctx.build_octree(a.basecube, 12, pnt.shape[0], dynamic=dyn)
        assert n > 1 << 24
        pos, ang = a.poses(2, seed=5)
        lights = np.array([[900.0, 1500.0, 700.0], [300.0, 1300.0, 1200.0]], np.float32)
        for i in range(2):
            v = q.view(pos[i], ang[i], 321, 200, a.basecube, 12)
            for mask in (q.OUT_ALL, q.OUT_ALL | q.RENDER_COUNT):
                print(f"[case] {n} dynamic nodes, pose {i}, outputs {mask:#x}", flush=True)
                out = []
                for layout in (0, 1):
                    ctx.set_tuning(layout=layout)
                    ctx.render(v, lights, mask)
                    out.append(ctx.read_frame(0))
                    st = ctx.stats()
                    assert st["dual"] == 1 and st["compact"] == 1 - layout
                assert np.count_nonzero(out[0]["dyn"] > 0) > 1000
                for k in out[0]:
                    assert np.array_equal(out[0][k].view(np.uint8), out[1][k].view(np.uint8)), (i, mask, k)
