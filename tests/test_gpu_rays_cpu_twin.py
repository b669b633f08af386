"""Ray batches with the CPU twin's semantics at the sizes where their launch
changes shape (a share of less than a wave per wave, one ray per lane, the work
queue and the sharing after it), axis rays and rays from near the planes y = 0
and z = 0 among them: status, leaf and entry point bits equal the oracle's."""
import numpy as np
import pytest

import qubatron_amd as q
from oracle import pyoracle as po
from tests import helpers as H
from tests.test_host_sem import axis_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene():
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    ctx = q.Context(0)
    ctx.upload_octree(nodes)
    ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    rng = np.random.default_rng(31)
    n = 400003
    org = rng.uniform(20.0, 1780.0, (n, 3)).astype(np.float32)
    dirs = rng.standard_normal((n, 3)).astype(np.float32)
    a = np.arange(0, n, 7)
    org[a], dirs[a] = axis_rays(rng, a.size)
    ref = po.OracleScene(nodes, None, None, sc.basecube, sc.depth).trace_many(org, dirs, semantics=po.SEM_CPU)
    yield ctx, sc, org, dirs, ref
    ctx.close()


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("n", [1, 65, 8191, 131071, 400003])
def test_cpu_twin_batches_equal_oracle(scene, n, layout):
    ctx, sc, org, dirs, ref = scene
    print(f"[case] {n} rays, layout {layout}", flush=True)
    ctx.set_tuning(layout=layout)
    got = ctx.trace_rays(org[:n], dirs[:n], sc.basecube, sc.depth, semantics=1)
    np.testing.assert_array_equal(got["status"], ref["status"][:n])
    np.testing.assert_array_equal(got["leaf"], ref["leaf"][:n])
    hit = got["status"] == 1
    np.testing.assert_array_equal(got["isp"][hit].view(np.uint32), ref["isp"][:n][hit].view(np.uint32))
    assert (got["model"][hit] >= 0).all() and (got["model"][~hit] == -1).all()
