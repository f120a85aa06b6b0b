"""CPU: the hull builder's 32-bit orientation test (csrc/hull_orient.h,
compiled here for the host) against 64 bits.  What it is sure of must be
right at every size of the coordinates: the volume is of cubic size, so it
overflows from about 5e12 on and underflows below 1e-15."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mind-fcl_amd", "csrc")
WRAP = """#include "hull_orient.h"
extern "C" void decide(const float* p, long n, int* out) {
  for (long i = 0; i < n; ++i, p += 12) out[i] = mfcl::sees32(mfcl::planeOf(p, p + 3, p + 6), p + 9);
}
"""


@pytest.fixture(scope="module")
def decide(tmp_path_factory):
    d = tmp_path_factory.mktemp("orient")
    (d / "w.cpp").write_text(WRAP)
    so = str(d / "w.so")
    # the device code is compiled without fused multiply-adds too (dmath.h)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                           str(d / "w.cpp"), "-o", so])
    lib = C.CDLL(so)

    def run(p):
        p = np.ascontiguousarray(p, np.float32)
        out = np.zeros(len(p), np.int32)
        lib.decide(p.ctypes.data_as(C.c_void_p), C.c_long(len(p)), out.ctypes.data_as(C.c_void_p))
        return out

    return run


@pytest.mark.parametrize("size", [1e-30, 1e-15, 1e-12, 1e-3, 1.0, 1e6, 3e12, 7e12, 1e13, 2e13, 1e14, 1e18, 1e25, 1e38])
def test_sure_decisions_are_right(decide, size):
    rng = np.random.default_rng(int(abs(np.log10(size)) * 10) + 3)
    p = (rng.normal(size=(400000, 4, 3)) * size * rng.uniform(0.05, 1, (400000, 1, 1))).clip(-3e38, 3e38)
    # a third of the points close to their face's plane
    near = slice(0, 400000, 3)
    w = rng.dirichlet((1, 1, 1), len(p[near]))[..., None]
    p[near, 3] = (p[near, :3] * w).sum(1) * (1 + rng.normal(scale=1e-6, size=(len(w), 1)))
    p = p.astype(np.float32)
    got = decide(p)
    # 64 bits: no overflow (coordinates of at most 3.4e38, their cube 4e115)
    q = p.astype(np.float64)
    u, v, x = q[:, 1] - q[:, 0], q[:, 2] - q[:, 0], q[:, 3] - q[:, 0]
    vol = (np.cross(u, v) * x).sum(1)
    sure = got >= 0
    assert np.array_equal(got[sure] == 1, vol[sure] > 0)
    if 1e-3 <= size <= 1e6:  # a filter that decides nothing would pass too
        far = np.ones(len(p), bool)
        far[near] = False
        assert sure[far].mean() > 0.999


def test_not_finite_is_not_sure(decide):
    base = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0.2, 0.2, 1]], np.float32)
    sets = []
    for bad in (np.inf, -np.inf, np.nan):
        for i in range(4):
            for k in range(3):
                p = base.copy()
                p[i, k] = bad
                sets.append(p)
    assert (decide(np.array(sets)) == -1).all()
    assert decide(base[None])[0] == 1
