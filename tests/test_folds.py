"""The fold test of a surface (h2lib_amd/csrc/folds.h) against all pairs of
triangles at each vertex, and its work at vertices of many triangles (CPU)."""
import ctypes as C
import os
import shutil
import subprocess
import time

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "h2lib_amd", "csrc")


@pytest.fixture(scope="module")
def folds(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("folds")
    src, lib = str(d / "folds.cpp"), str(d / "folds.so")
    with open(src, "w") as f:
        f.write('#include "folds.h"\n'
                'extern "C" int folds(uint32_t nv, const uint32_t *p,\n'
                '                     const uint32_t *t, const double *n) {\n'
                '  return h2hip::folds(nv, p, t, n);\n}\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    "-ffp-contract=off", "-I", CSRC, src, "-o", lib],
                   check=True)
    f = C.CDLL(lib).folds

    def call(normals):
        """One vertex with these triangles."""
        n = np.ascontiguousarray(normals, dtype=np.float64)
        ptr = np.array([0, len(n)], dtype=np.uint32)
        tri = np.arange(len(n), dtype=np.uint32)
        return bool(f(1, ptr.ctypes.data_as(C.c_void_p),
                      tri.ctypes.data_as(C.c_void_p),
                      n.ctypes.data_as(C.c_void_p)))
    return call


def all_pairs(n):
    g = n @ n.T
    d = np.diag(g)
    with np.errstate(invalid="ignore"):
        return bool(((g < 0) & (g * g > 0.9 * d[:, None] * d[None, :])).any())


@pytest.mark.parametrize("count", [1, 2, 6, 32, 33, 64, 300])
def test_same_as_all_pairs(folds, count):
    rng = np.random.default_rng(count)
    seen = set()
    for trial in range(400):
        # normals within a cap, and some near the opposite of one of them at
        # 10 to 30 degrees (the line lies at acos(sqrt(0.9)) = 18.4)
        axis = rng.normal(size=3)
        n = axis / np.linalg.norm(axis) + 0.2 * rng.normal(size=(count, 3))
        if trial % 2 and count > 1:
            a = n[rng.integers(count)]
            t = np.cross(a, rng.normal(size=3))
            ang = np.radians(rng.uniform(10.0, 30.0))
            n[rng.integers(count)] = -(
                np.cos(ang) * a / np.linalg.norm(a) +
                np.sin(ang) * t / np.linalg.norm(t))
        if trial % 3 == 0:
            n *= 10.0 ** rng.uniform(-3, 3, size=(count, 1))
        if trial % 7 == 0:
            n[rng.integers(count)] = rng.choice([0.0, np.nan])
        want = all_pairs(n)
        seen.add(want)
        assert folds(n) == want, (count, trial)
    assert seen == ({False} if count == 1 else {False, True})


def test_work_at_vertices_of_many_triangles(folds):
    m = 200000
    ang = 2.0 * np.pi * np.arange(m) / m

    def cone(half):
        h = np.radians(half)
        return np.stack([np.cos(ang) * np.cos(h), np.sin(ang) * np.cos(h),
                         np.full(m, np.sin(h))], 1)
    t0 = time.perf_counter()
    assert not folds(np.tile([0.0, 0.0, 1.0], (m, 1)))  # a flat fan
    assert not folds(cone(60.0))
    assert folds(cone(5.0))
    assert folds(cone(12.0))  # (not opposite: its candidates are too many)
    # (2e10 comparisons each when every pair is compared)
    assert time.perf_counter() - t0 < 5.0
