"""bs_metrics against a brute-force restatement at the sizes where the cell
search can go wrong: fewer than three cells per axis, boids at the field's
faces, sparse flocks whose nearest neighbour lies rings away, more links per
boid than a lane collects, and more boids than one workgroup's."""
import numpy as np
import pytest

import boidssimulatormpi_amd as B
from boidssimulatormpi_amd import engine as E

pytestmark = pytest.mark.gpu


def brute(pos, vel, F, eps, min_size):
    n = len(pos)
    d = np.abs(pos[:, None] - pos[None])
    d = np.minimum(d, F - d)
    s = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
    np.fill_diagonal(s, np.inf)
    label = np.arange(n)
    link = s < eps * eps
    while True:
        new = np.minimum(label, np.where(link, label[None], n).min(1))
        new = np.minimum(new, new[new])
        if np.array_equal(new, label):
            break
        label = new
    size = np.bincount(label, minlength=n)
    u = vel / np.linalg.norm(vel, axis=1, keepdims=True)
    return dict(polarisation=np.linalg.norm(u.sum(0)) / n, mean_nn=np.sqrt(s.min(1)).mean(),
                clusters=int(((size >= min_size) & (size > 0)).sum()), largest=int(size.max()))


@pytest.mark.parametrize("n,eps,shape", [
    (2, 0.3, "uniform"), (5, 0.9, "uniform"), (40, 0.49, "uniform"), (63, 0.02, "uniform"), (65, 0.34, "faces"),
    (257, 0.0, "sparse"), (1000, 0.05, "sparse"), (1500, 0.08, "faces"), (2049, 0.05, "clump"), (2500, 0.11, "uniform")])
def test_metrics_against_brute_force(n, eps, shape):
    F = 1.0
    g = np.random.default_rng(n)
    pos = g.random((n, 3))
    if shape == "faces":                           # within 1e-3 of a face, both sides
        pos = np.where(g.random((n, 3)) < 0.5, 1e-3 * pos, 1 - 1e-3 * pos)
        pos[: n // 2, 1:] = g.random((n // 2, 2))
    elif shape == "sparse":                        # a tight group and a few boids far from it
        pos[8:] = 0.5 + 0.02 * (pos[8:] - 0.5)
    elif shape == "clump":                         # dozens of links per boid
        pos = 0.3 + 0.2 * pos
    vel = 1e-3 * g.standard_normal((n, 3)) + 1e-4
    e = B.Engine(B.make_params(n, F, mode=E.MODE_ALLPAIRS_F64))
    e.set_state(pos=pos, vel=vel)
    for min_size in (1, 2, 7):
        got, want = e.metrics(eps, min_size), brute(pos, vel, F, eps, min_size)
        print(n, eps, shape, got, want, flush=True)
        assert (got["clusters"], got["largest"]) == (want["clusters"], want["largest"])
        # sums of n doubles below 1 in another order: n 2^-53 each
        assert abs(got["polarisation"] - want["polarisation"]) <= 4e-16 * n
        assert abs(got["mean_nn"] - want["mean_nn"]) <= 4e-16 * n
        assert e.metrics_noalloc(eps, min_size) == got
    e.close()


def test_metrics_workspace_grows_and_shrinks():
    # one engine's kept workspace serves calls of any size after it
    g = np.random.default_rng(1)
    n = 3000
    pos, vel = g.random((n, 3)), 1e-3 * g.standard_normal((n, 3))
    e = B.Engine(B.make_params(n, 1.0, mode=E.MODE_ALLPAIRS_F64))
    e.set_state(pos=pos, vel=vel)
    first = {eps: e.metrics(eps) for eps in (0.5, 0.01, 0.2)}       # 1, 14 and 4 cells per axis
    assert {eps: e.metrics(eps) for eps in (0.01, 0.2, 0.5)} == first
    e.close()
