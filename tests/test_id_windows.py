"""The windows of ids in which crowded owners of the float grid take their
boids: every boid once, in ascending id, in few passes however the ids of the
boids in reach are spread."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
CAP = 1024


@pytest.fixture(scope="module")
def passes(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("probe") / "windows.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "boidssimulatormpi_amd", "csrc"), "-o", so,
                    os.path.join(ROOT, "tests", "windows_probe.cpp")], check=True)
    f = ctypes.CDLL(so).window_passes
    f.restype = ctypes.c_int64

    def count(ids, n):
        ids = np.unique(ids).astype(np.uint32)
        return f(ids.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), len(ids), n, CAP), len(ids)
    return count


def spreads(n, m, g):
    if n < 1 << 28:
        yield "random", g.choice(n, m, replace=False)
        yield "clump and dust", np.concatenate([np.arange(n // 3, n // 3 + m // 2), g.choice(n, m // 2, replace=False)])
    yield "first", np.arange(m)
    yield "last", np.arange(n - m, n)
    yield "middle", np.arange(n // 2, min(n, n // 2 + m))
    yield "every third", np.arange(0, min(n, 3 * m), 3)
    yield "two clumps", np.concatenate([np.arange(n // 4, n // 4 + m // 2), np.arange(3 * n // 4 - m // 2, 3 * n // 4)])


@pytest.mark.parametrize("n", [1025, 4096, 8192, 65536, 1 << 20, 1 << 24, 1 << 28])
def test_windows_cover_in_few_passes(passes, n):
    g = np.random.default_rng(n)
    for m in (1, CAP, CAP + 1, 1500, 4000, 8000, 60000):
        if m > n:
            continue
        for name, ids in spreads(n, m, g):
            k, m_ = passes(ids, n)
            # m_ / 768 windows, each met once and at most once too wide; around each of two clumps the width comes
            # down from n at least fourfold a pass (found / 768 >= 4 while a clump of 3072 or more overflows, half
            # at worst) and goes up fourfold
            most = 1 if m_ <= CAP else 2 * (m_ // (CAP * 3 // 4) + 1) + 4 * int(np.log2(n))
            assert 0 < k <= most, (n, m, name, k)
