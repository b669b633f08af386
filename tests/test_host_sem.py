"""Sharing of rays between the lanes of a wave (qubatron_amd/csrc/device/split.hpp)
with the CPU twin's and the particle pass's semantics, compiled for the host:
status, leaf and entry point bits equal the oracle's serial trace, axis rays
and rays near the planes y = 0 and z = 0 among them (the plane tests' defaults
for a zero direction differ between the semantics)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import qubatron_amd as q
from oracle import pyoracle as po
from tests.test_host_trace import rays

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BC = np.array([0.0, 1800.0, 1800.0, 1800.0], np.float32)


@pytest.fixture(scope="module")
def hs(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hostsem") / "libhostsem.so")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-Wno-unknown-pragmas",
           "-Wno-enum-compare", "-I" + os.path.join(ROOT, "tests", "hosttrace"),
           "-I" + os.path.join(ROOT, "qubatron_amd", "csrc", "device"), "-o", out,
           os.path.join(ROOT, "tests", "hosttrace", "host_sem.cpp")]
    subprocess.run(cmd, check=True)
    lib = C.CDLL(out)
    f32p, i32p = C.POINTER(C.c_float), C.POINTER(C.c_int32)
    lib.ht_sem.argtypes = [i32p, C.c_size_t, f32p, C.c_int, C.c_int, C.c_int, C.c_int, f32p, f32p, C.c_size_t, C.c_int,
                           i32p, i32p, f32p]
    return lib


def axis_rays(rng, n):
    """Rays along the axes and in the axis planes, some from points close to y = 0 and z = 0."""
    org = rng.uniform(1.0, 1799.0, (n, 3)).astype(np.float32)
    org[::3, 1] = rng.uniform(-2.0, 2.0, org[::3].shape[0])
    org[1::3, 2] = rng.uniform(-2.0, 2.0, org[1::3].shape[0])
    d = rng.standard_normal((n, 3)).astype(np.float32)
    d[np.arange(n), rng.integers(0, 3, n)] = 0.0
    two = np.arange(0, n, 2)
    d[two, rng.integers(0, 3, two.size)] = 0.0
    return org, d


@pytest.mark.parametrize("sem,layout", [(1, 0), (1, 1), (2, 0)])
@pytest.mark.parametrize("levels,npts", [(2, 30), (7, 6000), (12, 30000)])
@pytest.mark.parametrize("per_wave", [1, 9, 64])
def test_split_equals_serial(hs, levels, npts, per_wave, sem, layout):
    rng = np.random.default_rng(levels * 100 + per_wave + sem)
    pts = rng.uniform(1.0, 1799.0, (npts, 3)).astype(np.float32)
    nodes = np.ascontiguousarray(q.octree_from_points(pts, BC, levels).nodes(), np.int32)
    a, b = rays(rng, 90), axis_rays(rng, 90)
    org, dirs = (np.ascontiguousarray(np.vstack([x, y]), np.float32) for x, y in zip(a, b))
    ref = po.OracleScene(nodes, None, None, BC, levels).trace_many(org, dirs,
                                                                   semantics=po.SEM_CPU if sem == 1 else po.SEM_PARTICLE)
    n = org.shape[0]
    i32 = lambda x: x.ctypes.data_as(C.POINTER(C.c_int32))
    f32 = lambda x: x.ctypes.data_as(C.POINTER(C.c_float))
    for grid in (0, 1):
        st, lf, isp = np.empty(n, np.int32), np.empty(n, np.int32), np.empty((n, 4), np.float32)
        assert hs.ht_sem(i32(nodes), nodes.shape[0], f32(BC), levels, layout, sem, grid, f32(org), f32(dirs), n, per_wave,
                         i32(st), i32(lf), f32(isp)) == 0
        what = f"grid {grid}"
        np.testing.assert_array_equal(st, ref["status"], err_msg=what)
        np.testing.assert_array_equal(lf, ref["leaf"], err_msg=what)
        np.testing.assert_array_equal(isp.view(np.uint32), ref["isp"].view(np.uint32), err_msg=what)
