"""The cells of a row that the metrics' ring search reads: each of the run's
once, around the field's faces too (a side cell that wrapped used to bring the
cells up to the face with it)."""
import ctypes
import os
import subprocess

import numpy as np

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))


def test_runs_name_their_cells_once(tmp_path):
    so = str(tmp_path / "ring.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "boidssimulatormpi_amd", "csrc"), "-o", so,
                    os.path.join(ROOT, "tests", "ring_probe.cpp")], check=True)
    f = ctypes.CDLL(so).run_cells
    for G in (1, 2, 3, 4, 5, 8, 13):
        out = np.zeros(4 * G, np.int32)
        for x0 in range(1 - G, 2 * G):
            for x1 in range(x0, min(x0 + G - 1, 2 * G)):           # fewer than G cells
                n = f(x0, x1, G, out.ctypes.data_as(ctypes.c_void_p))
                assert sorted(out[:n]) == sorted(x % G for x in range(x0, x1 + 1)), (G, x0, x1)
        n = f(0, G - 1, G, out.ctypes.data_as(ctypes.c_void_p))    # a whole row
        assert list(out[:n]) == list(range(G))
