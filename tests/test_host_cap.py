"""The iteration cap of the traversal (qubatron_amd/csrc/device/trace.hpp,
split.hpp), compiled for the host: a ray is aborted exactly when its serial
trace takes more steps than the cap, and has the uncapped result otherwise,
traced alone or shared between the lanes of a wave, on both layouts, with one
tree and two. The long rays run along a row of cells beside a row of points:
they enter every parent cell of the row and none of its leaves."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import qubatron_amd as q
from tests.test_host_trace import oracle_trace, rays

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BC = (0.0, 4096.0, 4096.0, 4096.0)
LEVELS = 12  # leaves of edge 1
ABORT = -2


@pytest.fixture(scope="module")
def hc(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hostcap") / "libhostcap.so")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-Wno-unknown-pragmas",
           "-Wno-enum-compare", "-I" + os.path.join(ROOT, "tests", "hosttrace"),
           "-I" + os.path.join(ROOT, "qubatron_amd", "csrc", "device"), "-o", out,
           os.path.join(ROOT, "tests", "hosttrace", "host_cap.cpp")]
    subprocess.run(cmd, check=True)
    lib = C.CDLL(out)
    f32p, i32p = C.POINTER(C.c_float), C.POINTER(C.c_int32)
    lib.ht_cap.argtypes = [i32p, C.c_size_t, i32p, C.c_size_t, f32p, C.c_int, C.c_int, C.c_int, f32p, f32p, C.c_size_t,
                           C.c_int, C.c_int, i32p, i32p, f32p, C.POINTER(C.c_int64)]
    return lib


@pytest.fixture(scope="module")
def scene():
    """Points beside the rays (y0 + 1 is the other row of the same parents) and a leaf at the far end; rays along x,
    a little tilted, and random ones."""
    rng = np.random.default_rng(11)
    x = np.arange(0.5, 4088.0, 2.0)
    row = lambda y, z: np.stack([x, np.full_like(x, y), np.full_like(x, z)], 1)
    pts = np.concatenate([row(101.5, 100.5), row(100.5, 101.5), row(103.5, 100.5), [[4094.5, 100.5, 100.5]],
                          rng.uniform(1.0, 4095.0, (300, 3))]).astype(np.float32)
    nodes = np.ascontiguousarray(q.octree_from_points(pts, BC, LEVELS).nodes())
    dyn = np.ascontiguousarray(q.octree_from_points((row(101.5, 101.5) + [1.0, 0.0, 0.0]).astype(np.float32), BC,
                                                    LEVELS).nodes())
    n = 6
    org = np.stack([rng.uniform(-50.0, 700.0, n), rng.uniform(100.3, 100.7, n), rng.uniform(100.3, 100.7, n)], 1)
    d = np.stack([np.ones(n), rng.uniform(-5e-5, 5e-5, n), rng.uniform(-5e-5, 5e-5, n)], 1)
    d[::2, 1:] = np.float32(1e-6)
    o2, d2 = rays(rng, 6)
    return (nodes, dyn, np.ascontiguousarray(np.vstack([org, o2]), np.float32),
            np.ascontiguousarray(np.vstack([d, d2]), np.float32))


@pytest.mark.parametrize("per_wave", [0, 2, 64])
@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("layout", [0, 1])
def test_cap_is_exact(hc, scene, layout, dual, per_wave):
    nodes, dyn, org, dirs = scene
    dyn = dyn if dual else None
    ref = oracle_trace(nodes, BC, LEVELS, org, dirs, dyn)
    n, bc = org.shape[0], np.asarray(BC, np.float32)
    i32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))
    f32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))

    def go(cap, grid):
        st, lf, isp, steps = np.empty(n, np.int32), np.empty(n, np.int32), np.empty((n, 4), np.float32), np.empty(n, np.int64)
        assert hc.ht_cap(i32(nodes), nodes.shape[0], i32(dyn) if dual else None, dyn.shape[0] if dual else 0, f32(bc),
                         LEVELS, layout, grid, f32(org), f32(dirs), n, cap, per_wave, i32(st), i32(lf), f32(isp),
                         steps.ctypes.data_as(C.POINTER(C.c_int64))) == 0
        return st, lf, isp, steps

    steps = go(1 << 22, 1)[3]
    assert steps.max() > 3000 and (steps > 1100).sum() > 4
    # whole from the start (below 1024), one round of sharing or a few and then whole, and sharing to the end
    caps = [1, 5, 100, 1024, 2047, 2048, int(steps.max()) - 1, int(steps.max()), 9000, 100000, int(np.median(steps))]
    for k, cap in enumerate(caps):
        st, lf, isp, ns = go(cap, k & 1)
        np.testing.assert_array_equal(ns, steps)
        over = steps > cap
        what = f"cap {cap}"
        np.testing.assert_array_equal(st, np.where(over, ABORT, ref["status"]), err_msg=what)
        np.testing.assert_array_equal(lf[~over], ref["leaf"][~over], err_msg=what)
        np.testing.assert_array_equal(isp[~over].view(np.uint32), ref["isp"][~over].view(np.uint32), err_msg=what)
