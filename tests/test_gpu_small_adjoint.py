"""The one-launch adjoint and fused steps at the edges of their rows, passes and
target counts: the cotangents against 64 bits, the fused forward part bit-equal
to the one-launch forward step.

A term carries at most 40 roundings of 2^-24 (differences of x and g, d, K, q,
r . h, the vector) of its largest part, its sum n / 256 + 12 more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _cfg(count, info):
    return next(c for c in range(count()) if info(c)["block"] == 1024)


@pytest.mark.parametrize("n", [1, 2, 15, 17, 64, 65, 257, 511, 513, 1024, 1025, 2048, 2049, 2600])
@pytest.mark.parametrize("eps", [1e-3, 0.0])
def test_small_adjoint(nb, gpu, n, eps):
    import torch

    acfg = _cfg(nb.adjoint_config_count, nb.adjoint_config_info)
    fcfg = _cfg(nb.forward_config_count, nb.forward_config_info)
    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    p = nb.default_params(num_particles=n, G=1.0 / n, dist_eps=eps)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    gen = torch.Generator().manual_seed(n)
    lxn, lvn = (torch.randn(3, n, generator=gen).to(gpu) for _ in range(2))
    dt, G = float(np.float32(p.dt)), float(np.float32(p.G))
    X, LX, LV = P.double(), lxn.double(), lvn.double()
    g = LV + dt * LX
    r = X[:, None, :] - X[:, :, None]
    h = g[:, None, :] - g[:, :, None]
    d = (r * r).sum(0) + float(np.float32(eps))
    K, q = d ** -1.5, 1.0 / d
    K.fill_diagonal_(0.0)
    q.fill_diagonal_(0.0)
    rh = (r * h).sum(0)
    lx = LX + dt * G * (K * (h - 3.0 * rh * q * r)).sum(2)
    size = g.abs()[:, None, :] + g.abs()[:, :, None]
    mag = (K * (size + 3.0 * (r.abs() * size).sum(0) * q * r.abs())).sum(2)
    bound = U * ((40 + n / 256 + 12) * dt * G * mag + 4 * (LX.abs() + lx.abs()))
    bv = U * 4 * (LV.abs() + dt * LX.abs())
    for fused in (False, True):
        ox, ov = torch.empty_like(P), torch.empty_like(P)
        v, N = V.clone(), torch.empty_like(P)
        if fused:
            nb.fwd_adjoint_step(p, P, v, N, lxn, lvn, ox, ov, cfg=acfg)
            v2, N2 = V.clone(), torch.empty_like(P)
            nb.forward_step(p, P, v2, N2, cfg=fcfg)
            assert torch.equal(v, v2) and torch.equal(N, N2)
        else:
            nb.adjoint_step(p, P, lxn, lvn, ox, ov, cfg=acfg)
        assert ((ox.double() - lx).abs() <= bound).all(), fused
        assert ((ov.double() - float(np.float32(p.damping)) * g).abs() <= bv).all(), fused
