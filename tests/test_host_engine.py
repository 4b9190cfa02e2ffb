"""The engine's host code -- transfers, staging, devices, chunk sizes -- over a stand-in for
the HIP runtime (host_runtime.cpp: several devices in host memory, kernels do
nothing, copies wait on their stream).  Each test runs in a process of its own,
which loads the stand-in ahead of the engine."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

PRELUDE = """
import ctypes, sys
import numpy as np
rt = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
for name in ("rt_device_bytes", "rt_in_flight", "rt_calls", "rt_copied_to"):
    getattr(rt, name).restype = ctypes.c_uint64
import boidssimulatormpi_amd as B
from boidssimulatormpi_amd import engine as E
L = B.lib()
RULES = dict(sep=(0.02, 0.75, 0.002), ali=(0.05, 0.75, 0.06), coh=(0.08, 0.75, 0.008), vmax=0.005, vmin=0.001)
F64 = ctypes.POINTER(ctypes.c_double)

def engine(n, device=0, mode=E.MODE_ALLPAIRS_F64, flags=E.FLAG_FORCES):
    e = B.Engine(B.make_params(n, 1.0, **RULES, mode=mode, flags=flags, device=device))
    assert rt.rt_calls(b"hipMalloc")               # the engine's calls end up in the stand-in
    return e

def state(n, seed=0):
    g = np.random.default_rng(seed)
    return g.random((n, 3)), g.random((n, 3))
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rt") / "host_runtime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(ROOT, "tests", "host_runtime.cpp")], check=True)
    return so


def drive(runtime, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), runtime], cwd=ROOT, text=True,
                       capture_output=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


# the staging's ways: one copy, several parts, pieces of several threads
SIZES = (1000, 30000, 400000)


def test_round_trip(runtime):
    # (the stand-in's kernels do nothing: what comes back is what the upload left in the transfer buffer)
    drive(runtime, f"""
    for n in {SIZES[1:]}:
        e = engine(n)
        for seed in (1, 2):
            p, v = state(n, seed)
            e.set_state(pos=p, vel=v)
            q, w = e.state_f64()
            assert np.array_equal(p, q) and np.array_equal(v, w), n
        assert not e.forces_f64().any()
        e.close()
    assert rt.rt_in_flight() == 0 and rt.rt_device_bytes(-1) == 0
    """)


@pytest.mark.parametrize("n", SIZES)
def test_engines_on_several_devices(runtime, n):
    # an engine works on its own device whatever the caller's is, which stays as it was
    drive(runtime, f"""
    n = {n}
    engines = [engine(n, device=k) for k in range(3)]
    for d in (3, 1):
        rt.hipSetDevice(d)
        for k, e in enumerate(engines):
            p, v = state(n, k)
            held = [rt.rt_device_bytes(j) for j in range(4)]
            e.set_state(pos=p, vel=v)
            e.step(2)
            q, w = e.state_f64()
            e.forces_f64()
            e.metrics(0.02)
            e.sync()
            assert rt.rt_current() == d
            assert [rt.rt_device_bytes(j) for j in range(4) if j != k] == [held[j] for j in range(4) if j != k]
            assert n < 11000 or np.array_equal(p, q) and np.array_equal(v, w)
    for e in engines:
        e.close()
    assert rt.rt_device_bytes(-1) == 0
    """)


@pytest.mark.parametrize("call", ["hipMemcpyAsync", "hipEventRecord", "hipEventSynchronize", "hipStreamSynchronize",
                                  "hipLaunchKernel"])
def test_failed_transfers_leave_no_copy_behind(runtime, call):
    # whichever call of a transfer fails, nothing still reads or writes the staging once it is lent again
    drive(runtime, f"""
    for n in {SIZES}:
        e = engine(n)
        p, v = state(n)
        failed = 0
        for op in (lambda: e.set_state(pos=p, vel=v), e.state_f64, e.forces_f64, e.state_f32):
            e.set_state(pos=p, vel=v)
            for k in range(1, 14):
                rt.rt_fail(b"{call}", k)
                try:
                    op()
                except B.EngineError as err:
                    failed += 1
                    assert "made to fail" in str(err)
                rt.rt_fail(b"{call}", 0)
                rt.hipGetLastError()
                assert rt.rt_in_flight() == 0, (n, k)
        assert failed or "Event" in "{call}" and n == 1000
        e.set_state(pos=p, vel=v)
        if n > 11000:
            q, w = e.state_f64()
            assert np.array_equal(p, q) and np.array_equal(v, w)
        e.close()
    assert rt.rt_device_bytes(-1) == 0
    """)


def test_transfers_without_memory_for_their_threads(runtime):
    # a large transfer whose helper threads cannot be made is carried by those that could, or by the caller
    drive(runtime, f"""
    n = {SIZES[2]}
    e = engine(n)
    p, v = state(n)
    q, w = np.empty_like(p), np.empty_like(v)
    at = [a.ctypes.data_as(F64) for a in (p, v, q, w)]
    e.set_state(pos=v, vel=p)
    for k in range(1, 7):
        rt.rt_fail_new(k)
        assert L.bs_set_state_f64(e._h, at[0], at[1]) == 0
        rt.rt_fail_new(k)
        assert L.bs_get_state_f64(e._h, at[2], at[3]) == 0
        rt.rt_fail_new(0)
        assert np.array_equal(p, q) and np.array_equal(v, w)
        p += 1.0
        v -= 1.0
    e.close()
    """)


@pytest.mark.parametrize("mode", [2, 3])
def test_chunk_size_as_reported(runtime, mode):
    # bs_info.fill is the chunk size in use and, passed back, gives the same engine
    drive(runtime, f"""
    from boidssimulatormpi_amd import autotune as T

    def grid(n, block, fill):
        F = max(1.0, (n / 16384.0) ** (1 / 3))
        e = B.Engine(B.make_params(n, F, **RULES, mode={mode}, block=block, fill=fill))
        assert e.info().mode == {mode}
        e.set_state(xyzv6=np.zeros((n, 6), np.float32))
        out = e.info().fill, e.grid()[0].chunk_boids
        e.close()
        return out
    for block in (0, 64, 128, 256):
        for n in (27, 1000, 13107, 16384, 20000, 32767, 32768, 50021, 131072, 600000):
            fill, boids = grid(n, block, 0)
            assert 10 <= fill <= 100 and boids == fill * (block or 64) // 100, (block, n)
            assert grid(n, block, fill) == (fill, boids)
        for fill in (10, 11, 24, 25, 60, 100):
            assert grid(3000, block, fill) == (fill, fill * (block or 64) // 100)
    for fill in (-1, 1, 9, 101):
        try:
            grid(3000, 0, fill)
        except B.EngineError as err:
            assert "10..100" in str(err)
        else:
            assert False, fill
    # the tuner times the engine's own choice too
    assert any(ps[0].fill == 0 for _, ps in T.candidates(B.make_params(3000, 1.0, **RULES, mode={mode})))
    """)


@pytest.mark.parametrize("n", [*SIZES, 12000, 130000])
def test_outputs_in_memory_the_runtime_knows(runtime, n):
    # Pinned arrays (above 1 MiB where they are two) and device arrays take the copies themselves: through the
    # staging they took up to 3.8 times as long (forces of 16384 boids 31 -> 119 us).
    drive(runtime, f"""
    n = {n}
    rt.rt_copied_to.argtypes = [ctypes.c_void_p]

    def block(make, count):
        p = ctypes.c_void_p()
        assert make(ctypes.byref(p), ctypes.c_size_t(8 * count), 0) == 0
        return p.value, np.frombuffer((ctypes.c_char * (8 * count)).from_address(p.value), np.float64)

    def at(a):
        return ctypes.cast(a, F64) if isinstance(a, int) else a.ctypes.data_as(F64)
    e = engine(n)
    pos, vel = state(n)
    e.set_state(pos=pos, vel=vel)
    for make, free in ((rt.hipHostMalloc, rt.hipHostFree), (rt.hipMalloc, rt.hipFree)):
        device = make is rt.hipMalloc
        (p, P), (v, V), (f, F) = (block(make, c * n) for c in (3, 3, 9))
        small = 48 * n <= 1 << 20 and not device
        for mine in ((p, v), (p, np.empty((n, 3))), (np.empty((n, 3)), v)):
            P[:] = V[:] = 0
            before = [rt.rt_copied_to(b) for b in (p, v)]
            assert L.bs_get_state_f64(e._h, at(mine[0]), at(mine[1])) == 0
            got = [rt.rt_copied_to(b) - c for b, c in zip((p, v), before)]
            known = [isinstance(m, int) for m in mine]
            want = [24 * n * (k and not small and (device or all(known))) for k in known]
            assert got == want, (device, known, got, want)
            if n > 11000:
                a, b = (P if known[0] else mine[0].ravel()), (V if known[1] else mine[1].ravel())
                assert np.array_equal(a, pos.ravel()) and np.array_equal(b, vel.ravel())
        F[:] = 1
        assert L.bs_get_forces_f64(e._h, at(f)) == 0
        assert rt.rt_copied_to(f) == 72 * n and not F.any()
        for b in (p, v, f):
            assert free(ctypes.c_void_p(b)) == 0
    e.close()
    """)


@pytest.mark.parametrize("n,parts", [(1000, 1), (16384, 1), (29127, 1), (29128, 3), (50021, 4), (116508, 6)])
def test_outputs_leave_in_few_parts(runtime, n, parts):
    # forces (72 bytes a boid) into pageable memory: up to 2 MiB one copy, then parts of about 1 MiB, 6 at most;
    # parts of 256 KiB took 1.5 times as long as the runtime's own copy (16384 boids 80 -> 116 us, one copy 68)
    drive(runtime, f"""
    e = engine({n})
    e.forces_f64()
    before = rt.rt_calls(b"hipMemcpyAsync")
    e.forces_f64()
    assert rt.rt_calls(b"hipMemcpyAsync") - before == {parts}, rt.rt_calls(b"hipMemcpyAsync") - before
    e.close()
    """)
