"""The pair kernels' work items and the sums of their partials where the number
of super-tiles makes them go wrong: one tile, one partial per run, a remainder
of the eight loads in flight, five workgroups per CU.  Every shape that takes
n, against the target-sharded one; a term carries at most 16 roundings of 2^-24
on each side and a sum n / 64 + 32 more (single sums of tiles and partials)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


@pytest.mark.parametrize("n", [127, 128, 129, 1024, 1025, 2049, 4100, 9800, 11521, 12801])
@pytest.mark.parametrize("acc", [0, 1])
def test_shapes_agree(nb, gpu, n, acc):
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    p = nb.default_params(num_particles=n, G=1.0 / n, dist_eps=1e-3)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    X, eps = P.double(), float(np.float32(1e-3))
    f, mag = torch.zeros_like(X), torch.zeros_like(X)
    for i0 in range(0, n, 512):
        r = X[:, None, :] - X[:, i0:i0 + 512, None]
        w = ((r * r).sum(0) + eps) ** -1.5
        f[:, i0:i0 + 512] = (r * w).sum(2)
        mag[:, i0:i0 + 512] = (r.abs() * w).sum(2)
    h = float(np.float32(p.dt)) * float(np.float32(p.G))
    v = V.double() * float(np.float32(p.damping)) + f * h
    bound = U * ((16 + n / 64 + 32) * mag * h + 4 * (v.abs() + mag * h))
    ran = 0
    for cfg in range(nb.forward_config_count()):
        if nb.forward_config_info(cfg)["scheme"] == "targets":
            continue
        v1, N = V.clone(), torch.empty_like(P)
        try:
            nb.forward_step(p, P, v1, N, cfg=cfg, acc=acc)
        except nb.NbError:
            assert acc == 1  # shapes without Kahan sums
            continue
        ran += 1
        assert ((v1.double() - v).abs() <= bound).all(), nb.forward_config_info(cfg)
    assert ran >= 4
