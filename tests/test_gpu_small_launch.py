"""The one-launch step for small systems at the edges of its rows (16 lanes),
passes (256 and 1024 sources) and target counts (4, 8 and 16 per workgroup).

A term carries at most 16 roundings of 2^-24 (differences, d, d^3, v_rsq_f32,
the product) and its sum n / 256 + 12 more (Kahan: 4), the update 4 of |v| and
|x|; the reference is the step in 64 bits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _cfg(nb):
    return next(c for c in range(nb.forward_config_count())
                if nb.forward_config_info(c)["block"] == 1024)


@pytest.mark.parametrize("n", [1, 2, 3, 15, 17, 64, 65, 255, 257, 1023, 1024, 1025, 2048, 2049,
                               4095, 4099])
@pytest.mark.parametrize("acc", [0, 1])
@pytest.mark.parametrize("eps", [1e-3, 0.0])
def test_small_launch(nb, gpu, n, acc, eps):
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    p = nb.default_params(num_particles=n, G=1.0 / n, dist_eps=eps)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    v0, N = V.double(), torch.empty_like(P)
    nb.forward_step(p, P, V, N, cfg=_cfg(nb), acc=acc)
    X = P.double()
    r = X[:, None, :] - X[:, :, None]
    d = (r * r).sum(0) + float(np.float32(eps))
    w = d ** -1.5
    w.fill_diagonal_(0.0)
    h = float(np.float32(p.dt)) * float(np.float32(p.G))
    f, mag = (r * w).sum(2) * h, (r.abs() * w).sum(2) * h
    damped = v0 * float(np.float32(p.damping))
    k = 16 + (4 if acc else n / 256 + 12)
    bv = U * (k * mag + 4 * (damped.abs() + mag))
    v = damped + f
    assert ((V.double() - v).abs() <= bv).all()
    dt = float(np.float32(p.dt))
    assert ((N.double() - (X + v * dt)).abs() <= bv * dt + 4 * U * (X.abs() + v.abs() * dt)).all()


def test_small_launch_predicated_and_nan(nb, gpu):
    import torch

    for n in (1, 700, 1500, 3000):
        pos, vel = nb.disk_ic(n)
        for eps in (1e-7, 0.0):
            out = []
            for cfg in (0, _cfg(nb)):
                p = nb.default_params(num_particles=n, calc_method=nb.NB_CALC_PREDICATED,
                                      dist_eps=eps)
                P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
                N = torch.empty_like(P)
                nb.forward_step(p, P, V, N, cfg=cfg)
                out.append((V.cpu().numpy(), N.cpu().numpy()))
            for a, b in zip(*out):
                assert np.array_equal(a, b, equal_nan=True)
        if n > 1:  # a NaN source reaches every target's force
            bad = [c.copy() for c in pos]
            bad[1][n // 2] = np.nan
            P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (bad, vel))
            N = torch.empty_like(P)
            nb.forward_step(nb.default_params(num_particles=n), P, V, N, cfg=_cfg(nb))
            assert torch.isnan(V).all()
