"""A build that runs out of device memory after its node array was allocated
(a max_device_bytes between the node array and the compact layout): the build
returns QBT_ENOMEM and leaves no tree, so renders, ray and particle batches
and downloads are refused instead of walking memory that nothing wrote, the
animated tree is left out of a frame, and a smaller build or an upload after
that gives the tree it would give in a new context."""
import numpy as np
import pytest

import qubatron_amd as q
from tests import helpers as H

pytestmark = pytest.mark.gpu
BIG = 1500000


def _cap(points, basecube, depth, setup, dynamic):
    """A limit under which `setup` and the upload of the points fit and the build of them gets its scratch (24 bytes a
    point and the sort's) and its node array, but not the whole compact layout (16 bytes a record and 4 a node)."""
    with q.Context(0) as c:
        setup(c)
        c.upload_points(points, dynamic=dynamic)
        held = c.device_bytes()
        n = c.build_octree(basecube, depth, points.shape[0], dynamic=dynamic)
    cap_nodes = n + n // 4 + 1024
    scratch = 24 * points.shape[0] + (48 << 20)  # the builder's smallest block, or the sort's own scratch
    layout = 16 * (n + n // 8 + 65536) + 4 * cap_nodes
    assert layout > 2 * (48 << 20)
    return held + scratch + 36 * cap_nodes + layout // 4, 36 * cap_nodes


def _fail(c, dynamic=False, array=0):
    """The build of BIG points fails, but its node array (`array` bytes) is there."""
    held = c.device_bytes()
    with pytest.raises(q.QbtError) as e:
        c.build_octree(np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32), 12, BIG, dynamic=dynamic)
    assert e.value.code == q._ffi.QBT_ENOMEM
    assert c.device_bytes() - held > array * 3 // 4


@pytest.mark.parametrize("before", ["nothing", "a tree"])
def test_static_build_out_of_memory(before):
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    big, _, _ = q.Scene(2, seed=3, npoints=BIG).points()

    def setup(c):
        c.upload_model(col, nrm)
        c.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
        if before == "a tree":
            c.upload_points(pnt)
            c.build_octree(sc.basecube, sc.depth, pnt.shape[0])

    cap, array = _cap(big, sc.basecube, 12, setup, False)
    v = q.view((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.basecube, sc.depth)
    with q.Context(0, max_device_bytes=cap) as c:
        setup(c)
        c.upload_points(big)
        print(f"[case] static build of {BIG} points under {cap} bytes, after {before}", flush=True)
        _fail(c, array=array)
        with pytest.raises(q.QbtError):
            c.render(v, sc.lights, q.OUT_ALL)
        with pytest.raises(q.QbtError):
            c.trace_rays(np.full((3, 3), 900.0, np.float32), np.ones((3, 3), np.float32), sc.basecube, 12)
        with pytest.raises(q.QbtError):
            c.particle_update(np.full((3, 3), 900.0, np.float32), np.ones((3, 3), np.float32), 12, 1800.0)
        with pytest.raises(q.QbtError):
            c.download_octree(1)
        print("[case] smaller build after the failure", flush=True)
        c.upload_points(pnt)
        assert c.build_octree(sc.basecube, sc.depth, pnt.shape[0]) == nodes.shape[0]
        assert np.array_equal(c.download_octree(nodes.shape[0]), nodes)
        c.render(v, sc.lights, q.OUT_ALL)
        g = c.read_frame(0)
        o = H.oracle_scene(1, npoints=100000).render((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.lights)
        mm = H.compare_frames(g, o)
        assert all(k == "exp" or x == 0 for k, x in mm.items()), mm


def test_refused_build_keeps_held_uploads(gpu_ctx):
    """A build refused for its points leaves the tree as it was, with the single-node uploads that the context still
    holds back."""
    bc = np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32)
    nodes = q.octree_from_points(np.random.default_rng(2).uniform(1, 1799, (500, 3)).astype(np.float32), bc, 6).nodes()
    gpu_ctx.upload_octree(nodes)
    edited = nodes.copy()
    i, o = np.argwhere(nodes[:, :8] > 0)[40]
    edited[i, o] = 0
    gpu_ctx.upload_octree(edited, start_node=int(i), end_node=int(i) + 1)
    gpu_ctx.upload_points(np.array([[-1000.0, 1000.0, 1000.0]], np.float32))  # an octet of -1
    with pytest.raises(q.QbtError) as e:
        gpu_ctx.build_octree(bc, 4, 1)
    assert e.value.code == q._ffi.QBT_ERANGE
    assert np.array_equal(gpu_ctx.download_octree(nodes.shape[0]), edited)


def test_upload_after_a_failed_build():
    """An array uploaded into the memory that the failed build allocated."""
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    big, _, _ = q.Scene(2, seed=3, npoints=BIG).points()

    def setup(c):
        c.upload_model(col, nrm)
        c.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)

    cap, array = _cap(big, sc.basecube, 12, setup, False)
    v = q.view((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.basecube, sc.depth)
    with q.Context(0, max_device_bytes=cap) as c:
        setup(c)
        c.upload_points(big)
        _fail(c, array=array)
        print("[case] whole upload after the failure", flush=True)
        c.upload_octree(nodes)
        c.render(v, sc.lights, q.OUT_ALL)
        g = c.read_frame(0)
        o = H.oracle_scene(1, npoints=100000).render((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.lights)
        mm = H.compare_frames(g, o)
        assert all(k == "exp" or x == 0 for k, x in mm.items()), mm


def test_dynamic_build_out_of_memory():
    """The frame after it shows the static tree alone, as with no animated tree."""
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    big, _, _ = q.Scene(2, seed=3, npoints=BIG).points()

    def setup(c):
        c.upload_model(col, nrm)
        c.upload_octree(nodes)

    cap, array = _cap(big, sc.basecube, 12, setup, True)
    v = q.view((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.basecube, sc.depth)
    with q.Context(0, max_device_bytes=cap) as c:
        setup(c)
        c.upload_points(big, dynamic=True)
        print(f"[case] dynamic build of {BIG} points under {cap} bytes", flush=True)
        _fail(c, dynamic=True, array=array)
        c.render(v, sc.lights, q.OUT_ALL)
        g = c.read_frame(0)
        assert c.stats()["dual"] == 0
        o = H.oracle_scene(1, npoints=100000).render((900.0, 900.0, 900.0), (np.pi, 0.0), 160, 120, sc.lights)
        mm = H.compare_frames(g, o)
        assert all(k == "exp" or x == 0 for k, x in mm.items()), mm
