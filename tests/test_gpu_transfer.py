"""States and forces in and out of an engine at the sizes where the transfer
changes its way: written by the kernel into pinned staging, copied through it
in one or several parts, and cut into
pieces that several threads carry (ragged last pieces, both arrays of a pair in
one piece)."""
import ctypes

import numpy as np
import pytest

import boidssimulatormpi_amd as B
from boidssimulatormpi_amd import engine as E

pytestmark = pytest.mark.gpu

# 512 KiB (kernel-written), 512 KiB and 256 KiB parts, 8 MiB in and out: from both sides
SIZES = [1, 7, 10922, 10923, 21845, 21846, 27307, 174762, 174763, 349525, 349526, 1000003]


@pytest.mark.parametrize("mode", [E.MODE_ALLPAIRS_F32REF, E.MODE_ALLPAIRS_F64, E.MODE_GRID_F64, E.MODE_GRID_MIXED,
                                  E.MODE_GRID_F32REF])
@pytest.mark.parametrize("n", SIZES)
def test_state_round_trip(mode, n):
    g = np.random.default_rng(n)
    F = max(0.5, (n / 16384.0) ** (1 / 3))
    st = np.concatenate([F * 0.999 * g.random((n, 3)), 1e-3 * g.standard_normal((n, 3))], 1).astype(np.float32)
    print(mode, n, flush=True)
    e = B.Engine(B.make_params(n, F, mode=mode))
    for xyzv in (st, st[::-1].copy()):                 # the second one through used staging
        e.set_state(xyzv6=xyzv)
        p, v = e.state_f32()
        assert np.array_equal(p, xyzv[:, :3]) and np.array_equal(v, xyzv[:, 3:])
        p, v = e.state_f64()
        assert np.array_equal(p, xyzv[:, :3].astype(np.float64)) and np.array_equal(v, xyzv[:, 3:].astype(np.float64))
    if mode not in (E.MODE_ALLPAIRS_F32REF, E.MODE_GRID_F32REF):
        pos, vel = F * 0.999 * g.random((n, 3)), 1e-3 * g.standard_normal((n, 3))
        e.set_state(pos=pos, vel=vel)
        p, v = e.state_f64()
        assert np.array_equal(p, pos) and np.array_equal(v, vel)
        p, v = e.state_f32()
        assert np.array_equal(p, pos.astype(np.float32)) and np.array_equal(v, vel.astype(np.float32))
    e.close()


@pytest.mark.parametrize("n", [1000, 30000, 70001])
def test_forces_agree_between_types(n):
    F = (n / 16384.0) ** (1 / 3)
    st = B.generate_init(E.INIT_ISOTROPIC, n, F, 0.005, 0.001, seed=n)
    for mode in (E.MODE_GRID_F64, E.MODE_GRID_F32REF):
        e = B.Engine(B.make_params(n, F, mode=mode, flags=E.FLAG_FORCES))
        e.set_state(xyzv6=st)
        assert not e.forces_f64().any()                # zeros before the first update
        e.step(1)
        f64, f32 = e.forces_f64(), e.forces_f32()
        assert f64.any() and np.array_equal(f32, f64.astype(np.float32))
        e.close()


@pytest.mark.parametrize("n", [1000, 8000, 21845, 21846, 130000, 400000])
def test_outputs_into_pinned_memory(n):
    # staged (two arrays up to 1 MiB) and straight; one array of a pair pinned, the other not
    hip = ctypes.CDLL("libamdhip64.so")
    f64 = ctypes.POINTER(ctypes.c_double)
    F = max(1.0, (n / 16384.0) ** (1 / 3))
    g = np.random.default_rng(n)
    pos, vel = F * 0.999 * g.random((n, 3)), 1e-3 * g.standard_normal((n, 3))
    print(n, flush=True)
    for mode in (E.MODE_ALLPAIRS_F64, E.MODE_GRID_F64):
        e = B.Engine(B.make_params(n, F, mode=mode, flags=E.FLAG_FORCES))
        e.set_state(pos=pos, vel=vel)
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(72 * n), 0) == 0
        pin = np.frombuffer((ctypes.c_char * (72 * n)).from_address(p.value), np.float64)
        out = np.empty(9 * n)
        for a, b in ((pin[:3 * n], pin[3 * n:6 * n]), (pin[:3 * n], out[:3 * n]), (out[:3 * n], pin[:3 * n])):
            pin[:] = out[:] = np.nan
            assert B.lib().bs_get_state_f64(e._h, a.ctypes.data_as(f64), b.ctypes.data_as(f64)) == 0
            assert np.array_equal(a, pos.ravel()) and np.array_equal(b, vel.ravel())
        if mode == E.MODE_GRID_F64:
            e.step(1)
        pin[:] = np.nan
        assert B.lib().bs_get_forces_f64(e._h, pin.ctypes.data_as(f64)) == 0
        assert np.array_equal(pin, e.forces_f64().ravel())
        e.close()
        del pin
        assert hip.hipHostFree(p) == 0
