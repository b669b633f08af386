"""Sharing of rays between the lanes of a wave at the end of a launch
(qubatron_amd/csrc/device/split.hpp), compiled for the host and run on an
emulated 64-lane wave: status, leaf and entry point bits of every ray equal
the oracle's serial trace, for one to 64 rays a wave, both layouts, both cube
arithmetics, one and two trees, and a lane that starts a second ray.
"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import qubatron_amd as q
from tests import helpers as H
from tests.test_host_trace import oracle_trace, rays

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BC = (0.0, 1800.0, 1800.0, 1800.0)


@pytest.fixture(scope="module")
def hs(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hostsplit") / "libhostsplit.so")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-Wno-unknown-pragmas",
           "-Wno-enum-compare", "-I" + os.path.join(ROOT, "tests", "hosttrace"),
           "-I" + os.path.join(ROOT, "qubatron_amd", "csrc", "device"), "-o", out,
           os.path.join(ROOT, "tests", "hosttrace", "host_split.cpp")]
    subprocess.run(cmd, check=True)
    lib = C.CDLL(out)
    f32p, i32p = C.POINTER(C.c_float), C.POINTER(C.c_int32)
    lib.ht_split.argtypes = [i32p, C.c_size_t, i32p, C.c_size_t, f32p, C.c_int, C.c_int, C.c_int, f32p, f32p,
                             C.c_size_t, C.c_int, i32p, i32p, f32p]
    return lib


def check(lib, nodes, bc, levels, org, dirs, per_wave, dyn=None, grids=(0, 1)):
    ref = oracle_trace(nodes, bc, levels, org, dirs, dyn)
    nodes = np.ascontiguousarray(nodes, np.int32)
    org, dirs = np.ascontiguousarray(org, np.float32), np.ascontiguousarray(dirs, np.float32)
    n, bca = org.shape[0], np.asarray(bc, np.float32)
    i32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))
    f32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))
    d = np.ascontiguousarray(dyn, np.int32) if dyn is not None else None
    for layout in (0, 1):
        for grid in grids:
            st, lf, isp = np.empty(n, np.int32), np.empty(n, np.int32), np.empty((n, 4), np.float32)
            rc = lib.ht_split(i32(nodes), nodes.shape[0], i32(d) if d is not None else None,
                              0 if d is None else d.shape[0], f32(bca), levels, layout, grid, f32(org), f32(dirs), n,
                              per_wave, i32(st), i32(lf), f32(isp))
            what = f"layout {layout} grid {grid} rays per wave {per_wave}"
            assert rc == 0, what
            np.testing.assert_array_equal(st, ref["status"], err_msg=what)
            np.testing.assert_array_equal(lf, ref["leaf"], err_msg=what)
            np.testing.assert_array_equal(isp.view(np.uint32), ref["isp"].view(np.uint32), err_msg=what)


@pytest.mark.parametrize("levels,npts", [(1, 8), (2, 30), (4, 300), (9, 20000), (12, 30000)])
@pytest.mark.parametrize("per_wave", [1, 2, 17, 64])
def test_split_equals_serial(hs, levels, npts, per_wave):
    rng = np.random.default_rng(levels * 100 + per_wave)
    pts = rng.uniform(1.0, 1799.0, (npts, 3)).astype(np.float32)
    nodes = q.octree_from_points(pts, BC, levels).nodes()
    org, dirs = rays(rng, 160)
    check(hs, nodes, BC, levels, org, dirs, per_wave)


@pytest.mark.parametrize("per_wave", [1, 5, 33])
def test_split_scene_and_ties(hs, per_wave):
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=200000)
    rng = np.random.default_rng(5)
    org, dirs = rays(rng, 150, inside=1.0)
    # axis rays and rays from the mid-planes, and rays through the cube's corner lines
    org2 = np.array([[900, 900, 900]] * 6 + [[900, 1700, 900]] * 6, np.float32)
    d6 = np.array([[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1]], np.float32)
    org3 = np.array([[900, 900, 3000], [-100, 900, 900], [-5, -5, -5], [1801, 1801, 1801]], np.float32)
    d3 = np.array([[0, 0, -2100], [1890, -890, -890], [1, 1, 1], [-1, -1, -1]], np.float32)
    check(hs, nodes, sc.basecube, sc.depth, np.vstack([org, org2, org3]), np.vstack([dirs, d6, d6, d3]), per_wave)


@pytest.mark.parametrize("per_wave", [1, 9, 64])
def test_split_dual_tree(hs, per_wave):
    rng = np.random.default_rng(8)
    a = q.octree_from_points(rng.uniform(1, 1799, (3000, 3)).astype(np.float32), BC, 7).nodes()
    b = q.octree_from_points(rng.uniform(1, 1799, (500, 3)).astype(np.float32), BC, 7).nodes()
    org, dirs = rays(rng, 200)
    check(hs, a, BC, 7, org, dirs, per_wave, dyn=b)
