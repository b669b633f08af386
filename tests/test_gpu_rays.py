"""Ray and particle batches at the sizes where their launches change shape:
one ray, a wave and one more, a share of less than a wave per wave (the rays
are split over the idle lanes), one ray per lane, and several rays per lane
(the work queue). Status, leaf, model and entry point bits equal the oracle's
for every ray; particles equal theirs batch by batch."""
import numpy as np
import pytest

import qubatron_amd as q
from oracle import pyoracle as po
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene():
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    ctx = q.Context(0)
    ctx.upload_octree(nodes)
    ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    rng = np.random.default_rng(3)
    n = 700001
    org = rng.uniform(20.0, 1780.0, (n, 3)).astype(np.float32)
    dirs = rng.standard_normal((n, 3)).astype(np.float32)
    dirs[::97] *= np.array([1, 0, 0], np.float32)  # axis rays among them
    ref = po.OracleScene(nodes, None, None, sc.basecube, sc.depth).trace_many(org, dirs)
    yield ctx, sc, org, dirs, ref
    ctx.close()


@pytest.mark.parametrize("n", [1, 2, 63, 65, 2049, 8191, 131071, 393217, 700001])
def test_ray_batches_equal_oracle(scene, n):
    ctx, sc, org, dirs, ref = scene
    print(f"[case] {n} rays", flush=True)
    got = ctx.trace_rays(org[:n], dirs[:n], sc.basecube, sc.depth, semantics=0)
    np.testing.assert_array_equal(got["status"], ref["status"][:n])
    np.testing.assert_array_equal(got["leaf"], ref["leaf"][:n])
    hit = got["status"] == 1
    np.testing.assert_array_equal(got["isp"][hit].view(np.uint32), ref["isp"][:n][hit].view(np.uint32))
    assert (got["model"][hit] >= 0).all() and (got["model"][~hit] == -1).all()


@pytest.mark.parametrize("n", [1, 65, 4095, 400003])
def test_particle_batches_equal_small_batches(scene, n):
    """The result of a particle does not depend on the batch it is in (small batches are compared with the oracle in
    test_gpu_particles.py)."""
    ctx, sc, org, dirs, ref = scene
    print(f"[case] {n} particles", flush=True)
    spd = (dirs * 5.0).astype(np.float32)
    spd[::5, 0] = -100000.0
    p, v = ctx.particle_update(org[:n], spd[:n], sc.depth, float(sc.basecube[3]))
    for a in range(0, n, max(1, n // 3)):
        b = min(n, a + 61)
        ps, vs = ctx.particle_update(org[a:b], spd[a:b], sc.depth, float(sc.basecube[3]))
        np.testing.assert_array_equal(p[a:b].view(np.uint32), ps.view(np.uint32))
        np.testing.assert_array_equal(v[a:b].view(np.uint32), vs.view(np.uint32))
