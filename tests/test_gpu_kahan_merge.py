"""Kahan sums keep their compensation where the waves of a work item bring
theirs together."""
import numpy as np
import pytest

from test_gpu_forward import has_kahan

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def kahan_configs(nb):
    return [c for c in range(nb.forward_config_count())
            if nb.forward_config_info(c)["scheme"] != "targets"
            and has_kahan(nb.forward_config_info(c))]


@pytest.mark.parametrize("n", [3000, 4100, 10000])
@pytest.mark.parametrize("minus", [64, 32])
def test_cancelling_waves(nb, gpu, n, minus):
    """All particles lie at the origin but for two groups of 16 at -+1 and one at
    2^11, in the sets of different waves (minus = 64; 32: in the part of one set
    that another wave takes, for the reaction sums).  Every sum is a multiple of
    2^-22 of at most 16 and every term an exact float, so a (sum, compensation)
    pair holds it exactly in any order: the force at the origin is 2^-22, which
    is below the rounding of the waves' sums of 16."""
    import torch

    x = np.zeros((3, n), np.float32)
    base = 1024
    x[0, base:base + 16] = 1.0
    x[0, base + minus:base + minus + 16] = -1.0
    x[0, base + minus + 16] = 2048.0
    p = nb.default_params(num_particles=n, G=1.0, dt=1.0, damping=1.0, dist_eps=1e-12)
    P = torch.from_numpy(x).to(gpu)
    at_origin = P[0] == 0
    for cfg in kahan_configs(nb):
        V, N = torch.zeros_like(P), torch.empty_like(P)
        nb.forward_step(p, P, V, N, cfg=cfg, acc=nb.NB_ACC_KAHAN)
        f = V[0][at_origin]
        # v_rsq_f32 is good to one unit
        assert ((f - 4 * U).abs() <= 2 * U * 4 * U).all(), (nb.forward_config_info(cfg), f)
        assert (V[1:, at_origin] == 0).all()


@pytest.mark.parametrize("n", [2049, 4100, 9800, 12801, 40959, 40960])
def test_error_does_not_grow_with_n(nb, gpu, n):
    """A term carries at most 16 roundings of 2^-24 (differences, d, d^3,
    v_rsq_f32, the product); its compensated sum, the rounding of a partial and
    the sums of partials 8 more, the update 4 of |v|."""
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    p = nb.default_params(num_particles=n, G=1.0 / n, dist_eps=1e-3)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    X, eps = P.double(), float(np.float32(1e-3))
    h = float(np.float32(p.dt)) * float(np.float32(p.G))
    idx = torch.arange(0, n, max(1, n // 2048), device=gpu)
    f = torch.empty(3, idx.numel(), dtype=torch.float64, device=gpu)
    mag = torch.empty_like(f)
    for k in range(0, idx.numel(), 256):
        r = X[:, None, :] - X[:, idx[k:k + 256], None]
        w = ((r * r).sum(0) + eps) ** -1.5
        f[:, k:k + 256] = (r * w).sum(2)
        mag[:, k:k + 256] = (r.abs() * w).sum(2)
    v = (V.double() * float(np.float32(p.damping)))[:, idx] + f * h
    bound = U * (24 * mag * h + 4 * (v.abs() + mag * h))
    for cfg in [-1] + (kahan_configs(nb) if n < 40000 else []):
        v1, N = V.clone(), torch.empty_like(P)
        nb.forward_step(p, P, v1, N, cfg=cfg, acc=nb.NB_ACC_KAHAN)
        assert ((v1[:, idx].double() - v).abs() <= bound).all(), (cfg, n)
