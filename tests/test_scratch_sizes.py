"""What a tile-pair step asks for is what its kernels write; the sizes that the
allocation-free step takes do not depend on it."""
import ctypes

import pytest


@pytest.mark.parametrize("n", [2049, 3327, 4097, 9727, 9728, 12800, 30001, 32767])
def test_trajectory_workspace_holds_the_partials(nb, n):
    """Workspace: positions (2), velocities, `every` position sets, two pairs of
    cotangents, and six sums per particle of ts^2 partials (ts (ts + 1) / 2 rows,
    ts (ts - 1) / 2 reactions) of a super-tile."""
    every = 3
    st = 256 if n >= 9728 else 128
    ts = -(-n // st)
    states = 3 * n * (3 + every + 4)
    assert nb.load().nb_traj_workspace_floats(n, every) == states + 6 * ts * ts * st


@pytest.mark.parametrize("n, acc, split", [(26625, 0, None), (37632, 0, None), (18817, 1, None),
                                           (26625, 0, 1), (18817, 0, 2)])
def test_noalloc_limits(nb, n, acc, split):
    """Refused before any use of the device or of the addresses."""
    cfg = -1 if split is None else next(
        c for c in range(nb.forward_config_count())
        if nb.forward_config_info(c)["scheme"] == "symmetric_tiles"
        and nb.forward_config_info(c)["unroll"] == 2
        and nb.forward_config_info(c)["split"] == split)
    p = nb.default_params(num_particles=n)
    rows = [0x1000000 * (k + 1) for k in range(9)]
    st = nb.load().nb_forward_step_noalloc_dev(ctypes.byref(p), *rows, n, cfg, acc, None)
    assert st == 5  # NB_ERR_UNSUPPORTED
    assert b"64 MiB" in nb.load().nb_last_error()
