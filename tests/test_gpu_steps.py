"""The reference-order steps (all-pairs, float grid) and the scan of the cell
counts at the sizes and positions where their ways change."""
import numpy as np
import pytest

import boidssimulatormpi_amd as B
from boidssimulatormpi_amd import engine as E
from oracle import oracle as O

from test_gpu_grid_build import check, single

pytestmark = pytest.mark.gpu

RULES = dict(sep=(0.02, 0.75, 0.002), ali=(0.05, 1.0, 0.06), coh=(0.05, 0.75, 0.008), vmax=0.005, vmin=0.001)


def flock(n, far, seed):
    """Boids of the field and, if far, clumps of them up to a thousand fields away, one without a position."""
    g = np.random.default_rng(seed)
    st = np.concatenate([g.random((n, 3)), 1e-3 * g.standard_normal((n, 3))], 1)
    st[::3, :3] = 0.5 + 0.03 * g.random((len(st[::3]), 3))
    if far and n > 8:
        at = g.choice([-1000.0, -3.1, -2.0, -1.01, 1.0, 1.99, 3.0, 1000.0], (n // 2, 3))
        st[: n // 2, :3] = at[np.arange(n // 2) // 4] + 0.02 * g.random((n // 2, 3))
        st[n // 4, 0] = np.nan
    return st


@pytest.mark.parametrize("mode", [E.MODE_ALLPAIRS_F32REF, E.MODE_ALLPAIRS_F64])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 1000, 3072, 3073, 4095, 4096, 4097, 5003])
@pytest.mark.parametrize("far", [False, True])
def test_allpairs_equals_oracle(mode, n, far):
    # one batch, several, and their remainders, up to 3072 and 4096 boids and beyond; lists
    # that fill in the middle of the flock
    print(mode, n, far, flush=True)
    f32 = mode == E.MODE_ALLPAIRS_F32REF
    st = flock(n, far, n)
    e = B.Engine(B.make_params(n, 1.0, **RULES, mode=mode, flags=E.FLAG_DIGEST))
    if f32:
        st = st.astype(np.float32)
        e.set_state(xyzv6=st)
    else:
        e.set_state(pos=st[:, :3].copy(), vel=st[:, 3:].copy())
    p, v = st[:, :3].copy(), st[:, 3:].copy()
    with np.errstate(invalid="ignore"):
        for t in range(2):
            _, d = O.step(O.params(1.0, **RULES), p, v, digest=True)
            e.step(1)
            gp, gv = e.state_f32() if f32 else e.state_f64()
            # the same operations in the same order
            assert np.array_equal(e.digest(), d), t
            assert np.array_equal(gp, p, equal_nan=True) and np.array_equal(gv, v, equal_nan=True), t
    e.close()


@pytest.mark.parametrize("n,cells", [(2, 3), (700, 3), (700, 4), (700, 16), (700, 17), (5000, 17), (4913, 17), (4912, 17)])
@pytest.mark.parametrize("out", [False, True])
def test_float_grid_half_and_whole_cells(n, cells, out):
    # half cells up to 16 cells per axis or n = 17^3, whole ones beyond; clumps
    # at the faces; boids a little outside the field (still within a cell edge of
    # all their neighbours)
    print(n, cells, out, flush=True)
    g = np.random.default_rng(n + cells)
    st = flock(n, False, n).astype(np.float32)
    edge = g.choice([0.0, 0.01, 0.98, 0.999], (n // 2, 3)) + 0.001 * g.random((n // 2, 3))
    st[: n // 2, :3] = edge
    st[0, 0] = 1.0
    if out:
        st[: n // 8, g.integers(3)] = np.float32(-0.004)
        st[n // 8: n // 4, g.integers(3)] = np.float32(1.004)
    flags = E.FLAG_DIGEST | E.FLAG_FORCES
    a = B.Engine(B.make_params(n, 1.0, **RULES, mode=E.MODE_ALLPAIRS_F32REF, flags=flags))
    b = B.Engine(B.make_params(n, 1.0, **RULES, mode=E.MODE_GRID_F32REF, flags=flags, cells_per_axis=cells))
    assert b.info().mode == E.MODE_GRID_F32REF and b.info().cells_per_axis == cells
    for again in range(2):                             # the second state starts anew
        for e in (a, b):
            e.set_state(xyzv6=st)
        for t in range(3):
            for e in (a, b):
                e.step(1)
            assert np.array_equal(a.digest(), b.digest()), t
            assert np.array_equal(a.forces_f32(), b.forces_f32()), t
            assert all(np.array_equal(x, y) for x, y in zip(a.state_f32(), b.state_f32())), t
        st = flock(n, False, n + 1).astype(np.float32)
    a.close()
    b.close()


@pytest.mark.parametrize("cells", [3, 12, 15, 16, 20, 25, 26, 31, 32, 33, 60, 150, 210])
def test_scan_sizes(cells):
    # one tile of 4096 counters, up to 4, up to 8, two launches, three launches
    n, rules = 3000, dict(RULES, sep=(0.002, 0.75, 0.002), ali=(0.002, 1.0, 0.06), coh=(0.002, 0.75, 0.008))
    print(cells, flush=True)
    e = B.Engine(B.make_params(n, 1.0, **rules, mode=E.MODE_GRID_F64, cells_per_axis=cells))
    e.set_state(xyzv6=np.abs(flock(n, False, cells)).astype(np.float32))
    for t in range(2):
        check(e, single(e, n, 1.0), f"{cells} cells per axis")
        e.step(1)
    e.close()


@pytest.mark.parametrize("mode", [E.MODE_GRID_F64, E.MODE_GRID_MIXED])
@pytest.mark.parametrize("n", [5, 1000, 13107, 16384, 32767, 32768])
def test_small_flocks_run_in_small_chunks(mode, n):
    # chunks of 6 boids, between 6 and 16, of 16 (their size never shows in the result)
    F = max(1.0, (n / 16384.0) ** (1 / 3))
    print(mode, n, flush=True)
    st = flock(n, False, n).astype(np.float32)
    a, b = (B.Engine(B.make_params(n, F, **RULES, mode=mode, flags=E.FLAG_DIGEST, fill=f)) for f in (0, 100))
    for e in (a, b):
        e.set_state(xyzv6=st)
    for t in range(3):
        for e in (a, b):
            e.step(1)
        check(a, single(a, n, F), f"n={n} update {t}")
        assert a.grid()[0].chunk_boids == 64 * max(10, 100 * n // (64 * 2048)) // 100
        assert np.array_equal(a.digest(), b.digest()), t
        assert all(np.array_equal(x, y) for x, y in zip(a.state_f64(), b.state_f64())), t
    a.close()
    b.close()


@pytest.mark.parametrize("spread", ["first", "middle", "two clumps", "clump and dust"])
def test_float_grid_crowds_of_neighbouring_ids(spread):
    # more boids within reach than an owner's list holds, their ids side by side: several windows of ids
    n, m = 9001, 2600
    print(spread, flush=True)
    g = np.random.default_rng(m)
    ids = {"first": np.arange(m), "middle": np.arange(n // 2, n // 2 + m),
           "two clumps": np.r_[1000: 1000 + m // 2, 7000: 7000 + m // 2],
           "clump and dust": np.r_[5000: 5000 + m // 2, g.choice(5000, m // 2, replace=False)]}[spread]
    st = flock(n, False, n).astype(np.float32)
    st[::3, :3] = g.random((len(st[::3]), 3))              # (no other crowd)
    st[ids, :3] = 0.4 + 0.01 * g.random((m, 3))
    flags = E.FLAG_DIGEST | E.FLAG_FORCES
    a = B.Engine(B.make_params(n, 1.0, **RULES, mode=E.MODE_ALLPAIRS_F32REF, flags=flags))
    b = B.Engine(B.make_params(n, 1.0, **RULES, mode=E.MODE_GRID_F32REF, flags=flags))
    assert b.info().mode == E.MODE_GRID_F32REF
    for e in (a, b):
        e.set_state(xyzv6=st)
    for t in range(2):
        for e in (a, b):
            e.step(1)
        assert t or ((a.digest()[ids, 0] >> 42) > 1024).all()          # alignment has no view cone here
        assert np.array_equal(a.digest(), b.digest()), t
        assert np.array_equal(a.forces_f32(), b.forces_f32()), t
        assert all(np.array_equal(x, y) for x, y in zip(a.state_f32(), b.state_f32())), t
    a.close()
    b.close()


@pytest.mark.parametrize("n", [1 << 18, (1 << 18) + 1])
def test_float_grid_at_the_largest_half_cells(n):
    # half cells up to 2^18 boids, whole ones beyond
    print(n, flush=True)
    F = (n / 16384.0) ** (1 / 3)
    st = B.generate_init(E.INIT_CLUSTERED, n, F, 0.005, 0.001, seed=3)
    a = B.Engine(B.make_params(n, F, **RULES, mode=E.MODE_ALLPAIRS_F32REF, flags=E.FLAG_DIGEST))
    b = B.Engine(B.make_params(n, F, **RULES, mode=E.MODE_GRID_F32REF, flags=E.FLAG_DIGEST))
    assert b.info().mode == E.MODE_GRID_F32REF
    for e in (a, b):
        e.set_state(xyzv6=st)
        e.step(1)
    assert np.array_equal(a.digest(), b.digest())
    assert all(np.array_equal(x, y) for x, y in zip(a.state_f32(), b.state_f32()))
    a.close()
    b.close()


@pytest.mark.parametrize("F", [1e-3, 3e-15, 1e-16, 1e-19, 3e-23, 1e-39, 1e5, 3e14, 1e16, 1e19, 1e39])
@pytest.mark.parametrize("mode", [E.MODE_ALLPAIRS_F32REF, E.MODE_GRID_F32REF, E.MODE_ALLPAIRS_F64])
def test_fields_of_any_size(mode, F):
    # fields whose squared lengths leave the floats' normal range are stepped without the candidate filter
    n = 1500
    print(mode, F, flush=True)
    if mode == E.MODE_GRID_F32REF and F < 1e-20:
        pytest.skip("squared distances underflow to 0: all-pairs then counts boids that no cell list meets")
    if mode == E.MODE_ALLPAIRS_F64:
        F = F ** 8 if 1e-39 < F < 1e39 else F                  # to 1e-184 and 1e152
    rules = {k: (v[0] * F, *v[1:]) for k, v in RULES.items() if k[0] != "v"}
    rules.update(vmax=0.005 * F, vmin=0.001 * F)
    st = flock(n, False, n)
    st[:, :3] = np.clip(st[:, :3], 0, 0.999)
    with np.errstate(all="ignore"):
        st = (st * F).astype(np.float32 if mode != E.MODE_ALLPAIRS_F64 else np.float64)
        st = np.where(np.isfinite(st), st, 0).astype(st.dtype)
        e = B.Engine(B.make_params(n, F, **rules, mode=mode, flags=E.FLAG_DIGEST))
        assert e.info().mode == mode
        p, v = st[:, :3].copy(), st[:, 3:].copy()
        e.set_state(xyzv6=st) if st.dtype == np.float32 else e.set_state(pos=p, vel=v)
        for t in range(2):
            _, d = O.step(O.params(F, **rules), p, v, digest=True)
            e.step(1)
            gp, gv = e.state_f32() if st.dtype == np.float32 else e.state_f64()
            assert np.array_equal(e.digest(), d), t
            assert np.array_equal(gp, p, equal_nan=True) and np.array_equal(gv, v, equal_nan=True), t
    e.close()
