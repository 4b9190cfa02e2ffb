"""The scan of the cell counts at the sizes where its way changes."""
import numpy as np
import pytest

import boidssimulatormpi_amd as B
from boidssimulatormpi_amd import engine as E

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
