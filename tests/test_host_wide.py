"""Both trees on their compact layouts where the dynamic one may have 2^24
records and more (qubatron_amd/csrc/device/trace.hpp, trace_step_c2), compiled
for the host with small trees: status, leaf and entry point bits of every ray
equal the oracle's, one by one and shared between the lanes of a wave."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import qubatron_amd as q
from tests.test_host_trace import oracle_trace, rays

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BC = (0.0, 1800.0, 1800.0, 1800.0)


@pytest.fixture(scope="module")
def hw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hostwide") / "libhostwide.so")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-Wno-unknown-pragmas",
           "-Wno-enum-compare", "-I" + os.path.join(ROOT, "tests", "hosttrace"),
           "-I" + os.path.join(ROOT, "qubatron_amd", "csrc", "device"), "-o", out,
           os.path.join(ROOT, "tests", "hosttrace", "host_wide.cpp")]
    subprocess.run(cmd, check=True)
    lib = C.CDLL(out)
    f32p, i32p = C.POINTER(C.c_float), C.POINTER(C.c_int32)
    lib.ht_wide.argtypes = [i32p, C.c_size_t, i32p, C.c_size_t, f32p, C.c_int, C.c_int, f32p, f32p, C.c_size_t, C.c_int,
                            i32p, i32p, f32p, C.POINTER(C.c_int64)]
    return lib


@pytest.mark.parametrize("levels,n,ndyn", [(1, 5, 3), (2, 60, 40), (7, 3000, 500), (7, 500, 20000), (11, 20000, 20000)])
@pytest.mark.parametrize("per_wave", [0, 1, 9, 64])
def test_wide_words_equal_oracle(hw, levels, n, ndyn, per_wave):
    rng = np.random.default_rng(levels * 10 + per_wave)
    a = np.ascontiguousarray(q.octree_from_points(rng.uniform(1, 1799, (n, 3)).astype(np.float32), BC, levels).nodes())
    b = np.ascontiguousarray(q.octree_from_points(rng.uniform(1, 1799, (ndyn, 3)).astype(np.float32), BC, levels).nodes())
    org, dirs = (np.ascontiguousarray(x, np.float32) for x in rays(rng, 300))
    ref = oracle_trace(a, BC, levels, org, dirs, b)
    bc = np.asarray(BC, np.float32)
    i32 = lambda x: x.ctypes.data_as(C.POINTER(C.c_int32))
    f32 = lambda x: x.ctypes.data_as(C.POINTER(C.c_float))
    m = org.shape[0]
    for grid in (0, 1):
        st, lf, isp, ex = np.empty(m, np.int32), np.empty(m, np.int32), np.empty((m, 4), np.float32), np.zeros(m, np.int64)
        assert hw.ht_wide(i32(a), a.shape[0], i32(b), b.shape[0], f32(bc), levels, grid, f32(org), f32(dirs), m, per_wave,
                          i32(st), i32(lf), f32(isp), ex.ctypes.data_as(C.POINTER(C.c_int64))) == 0
        np.testing.assert_array_equal(st, ref["status"])
        np.testing.assert_array_equal(lf, ref["leaf"])
        np.testing.assert_array_equal(isp.view(np.uint32), ref["isp"].view(np.uint32))
