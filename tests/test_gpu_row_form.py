"""The row form of the symmetric kernels (one wave holds a whole row
super-tile of 128, 256 or 512 particles, sources in sets of 64) at sizes
around its sets and super-tiles: last sets of 1 and 63 sources, super-tiles
with empty sets, one, two and three super-tiles.  Forward steps (plain and
Kahan sums) against the oracle step, adjoint and fused steps against the
fp64 adjoint."""
import numpy as np
import pytest

from test_gpu_forward import assert_step_parity, dev3, has_kahan

pytestmark = pytest.mark.gpu

SIZES = [63, 65, 127, 129, 191, 256, 257, 320, 513, 577, 1025]


def row_configs(count, info):
    """Shapes that run in the row form: tile pairs and super-tiles of 512."""
    return [c for c in range(count) if info(c)["scheme"] == "symmetric_tiles"
            or (info(c)["scheme"] == "symmetric" and info(c)["unroll"] == 2)]


@pytest.mark.parametrize("n", SIZES)
def test_row_form_forward(nb, orc, gpu, n):
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    params = nb.default_params(num_particles=n, G=1.0 / n)
    p = orc.params(num_particles=n, G=1.0 / n)
    ref, _ = orc.step_f32(p, pos, vel)
    for cfg in row_configs(nb.forward_config_count(), nb.forward_config_info):
        info = nb.forward_config_info(cfg)
        for acc in (nb.NB_ACC_PLAIN, nb.NB_ACC_KAHAN):
            if acc == nb.NB_ACC_KAHAN and not has_kahan(info):
                continue
            dp, dv = dev3(torch, pos, gpu), dev3(torch, vel, gpu)
            dn = [torch.empty_like(t) for t in dp]
            nb.forward_step(params, dp, dv, dn, cfg=cfg, acc=acc)
            torch.cuda.synchronize()
            assert_step_parity(orc, p, pos, vel, [t.cpu().numpy() for t in dn], ref,
                               np.arange(n), f"N={n} cfg {cfg} {info} acc {acc}")


@pytest.mark.parametrize("n", SIZES)
def test_row_form_adjoint(nb, orc, gpu, n):
    """fp32 rounding of about n / 2 terms of mixed sign per sum, against the
    sum's own size: 1e-5 (the bar of the other adjoint shape tests)."""
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    params = nb.default_params(num_particles=n, G=1.0, dt=1.0)
    p = orc.params(num_particles=n, G=1.0, dt=1.0)
    rng = np.random.default_rng(n)
    lxn, lvn = [rng.normal(size=(3, n)).astype(np.float32) for _ in range(2)]
    ref = np.stack(orc.adjoint_step_f64(p, np.stack(pos), lxn.astype(np.float64),
                                        lvn.astype(np.float64))[0])
    P, V, lxn, lvn = [torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel, lxn, lvn)]
    for cfg in row_configs(nb.adjoint_config_count(), nb.adjoint_config_info):
        for fused in (False, True):
            lx, lv, N = torch.empty_like(P), torch.empty_like(P), torch.empty_like(P)
            if fused:
                nb.fwd_adjoint_step(params, P, V.clone(), N, lxn, lvn, lx, lv, cfg=cfg)
            else:
                nb.adjoint_step(params, P, lxn, lvn, lx, lv, cfg=cfg)
            torch.cuda.synchronize()
            got = lx.double().cpu().numpy()
            err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            assert err <= 1e-5, (n, cfg, fused, err)
