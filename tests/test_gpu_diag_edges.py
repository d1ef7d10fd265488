"""fp64 diagnostics at the edges of their tiles and chunks (32 sources, 512
targets, 512 staged sources), and where the distance is zero or infinite.

Each term carries a few roundings of 2^-53 and a sum of N terms at most N
more, so |error| <= (N + 8) 2^-53 sum |term| against 80-bit sums.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _run(nb, gpu, pos, vel, eps, idx):
    import torch

    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    p = nb.default_params(num_particles=pos[0].size, G=1.0, dist_eps=eps)
    f = nb.forces_f64(p, P, torch.from_numpy(idx).to(gpu)).cpu().numpy()
    return f, nb.energy_momentum(p, P, V)


@pytest.mark.parametrize("n", [1, 2, 31, 33, 256, 257, 512, 513, 514, 1025, 2081])
@pytest.mark.parametrize("eps", [1e-7, 0.0])
def test_diag_edges(nb, gpu, n, eps):
    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    idx = np.unique(np.array([0, n // 2, n - 1, min(n - 1, 255), min(n - 1, 256)], np.int32))
    f, e = _run(nb, gpu, pos, vel, eps, idx)
    X = np.stack(pos).astype(np.longdouble)
    eps = np.longdouble(np.float32(eps))
    w = np.longdouble(0)
    for i in range(n):
        r = X[:, i + 1:] - X[:, i:i + 1]
        w += (1 / np.sqrt((r * r).sum(0) + eps)).sum()
    assert abs(e["potential"] + w) <= (n * n + 8) * U * w
    for k, i in enumerate(idx):
        r = np.delete(X, i, 1) - X[:, i:i + 1]
        d = (r * r).sum(0) + eps
        t = r / (d * np.sqrt(d))
        assert (abs(f[:, k] - t.sum(1)) <= (n + 8) * U * abs(t).sum(1)).all()
    V = np.stack(vel).astype(np.longdouble)
    assert abs(e["kinetic"] - 0.5 * (V * V).sum()) <= (n + 8) * U * 0.5 * (V * V).sum()
    assert (abs(np.array(e["momentum"]) - V.sum(1)) <= (n + 8) * U * abs(V).sum(1)).all()


def test_zero_and_infinite_distance(nb, gpu):
    n = 700
    pos, vel = nb.plummer_ic(n, seed=3, g_mass=1.0)
    idx = np.array([5, 6, 600], np.int32)
    pos = [np.array(c) for c in pos]
    same = [c.copy() for c in pos]
    for c in same:
        c[600] = c[5]
    f, e = _run(nb, gpu, same, vel, 0.0, idx)  # 0 * inf in both members' sums
    assert e["potential"] == -np.inf
    assert np.isnan(f[:, 0]).all() and np.isnan(f[:, 2]).all() and np.isfinite(f[:, 1]).all()
    far = [c.copy() for c in pos]
    far[0][600] = np.inf  # at an infinite distance: no potential, 0 * inf in x
    f, e = _run(nb, gpu, far, vel, 1e-7, idx)
    near = [np.delete(c, 600) for c in pos]
    g, h = _run(nb, gpu, near, [np.delete(c, 600) for c in vel], 1e-7, idx[:2])
    assert abs(e["potential"] - h["potential"]) <= 2 * n * n * U * abs(h["potential"])
    assert np.isnan(f[0]).all()
    # the others' y and z sums gain 0 from it
    assert np.allclose(f[1:, :2], g[1:], rtol=0, atol=1e-10 * abs(g).max())
