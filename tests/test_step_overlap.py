"""Steps whose outputs share memory with their sources: the one-launch shapes
write outputs while other workgroups still read sources, so such calls take a
shape of two launches by default and are refused when they name a one-launch
shape."""
import ctypes

import numpy as np
import pytest


def _one_launch(count, info):
    return next(c for c in range(count()) if info(c)["block"] == 1024)


def test_explicit_one_launch_refused(nb):
    """The check comes before any use of the device or of the addresses."""
    n, lib = 1000, nb.load()
    p = nb.default_params(num_particles=n)
    rows = [0x10000 * (k + 1) for k in range(21)]
    vecs = [rows[3 * k:3 * k + 3] for k in range(7)]

    def forward(pos, vel, nxt):
        return lib.nb_forward_step_dev(ctypes.byref(p), *pos, *vel, *nxt, n,
                                       _one_launch(nb.forward_config_count,
                                                   nb.forward_config_info), 0, None)

    def adjoint(*v):
        v = [nb.NbVec3(*r) for r in v]
        cfg = _one_launch(nb.adjoint_config_count, nb.adjoint_config_info)
        entry = lib.nb_adjoint_step_dev if len(v) == 5 else lib.nb_fwd_adjoint_step_dev
        return entry(ctypes.byref(p), *[ctypes.byref(r) for r in v], n, cfg, None)

    pos, vel, nxt, lxn, lvn, lx, lv = vecs
    shifted = [a + 4 * (n - 1) for a in pos]  # shares the last value of each row
    for bad in (pos, shifted, [lx[0], lx[1], pos[0]]):
        assert forward(pos, bad, nxt) == nb.NB_ERR_INVALID_ARG
        assert adjoint(pos, lxn, lvn, bad, lv) == nb.NB_ERR_INVALID_ARG
        assert adjoint(pos, lxn, lvn, lx, bad) == nb.NB_ERR_INVALID_ARG
        assert adjoint(pos, vel, nxt, lxn, lvn, bad, lv) == nb.NB_ERR_INVALID_ARG
    for src in (lxn, lvn):
        assert adjoint(pos, src, nxt, lxn, lvn, lx, lv) == nb.NB_ERR_INVALID_ARG
        assert adjoint(pos, vel, src, lxn, lvn, lx, lv) == nb.NB_ERR_INVALID_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 33, 1000, 1025, 2048])
def test_overlapping_steps(nb, gpu, n):
    """Bit-equal to the two-launch shape on separate arrays."""
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    p = nb.default_params(num_particles=n, G=1.0 / n)
    gen = torch.Generator().manual_seed(n)
    fixed = [torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel)]
    fixed += [torch.randn(3, n, generator=gen).to(gpu) for _ in range(2)]

    def fresh():
        P, V, X, W = [t.clone() for t in fixed]
        return P, V, X, W, [torch.empty_like(P) for _ in range(3)]

    def same(got, want):
        assert all(torch.equal(a, b) for a, b in zip(got, want))

    two = 8 if n < 1024 else 18
    P, V, X, W, (N, lx, lv) = fresh()
    nb.adjoint_step(p, P, X, W, lx, lv, cfg=two)
    want = lx, lv
    P, V, X, W, (N, lx, lv) = fresh()
    nb.adjoint_step(p, P, X, W, P, lv)
    same((P, lv), want)
    P, V, X, W, (N, lx, lv) = fresh()
    nb.adjoint_step(p, P, X, W, lx, P)
    same((lx, P), want)

    P, V, X, W, (N, lx, lv) = fresh()
    nb.fwd_adjoint_step(p, P, V, N, X, W, lx, lv, cfg=two)
    want = V, N, lx, lv
    P, V, X, W, (N, lx, lv) = fresh()
    nb.fwd_adjoint_step(p, P, V, X, X, W, lx, lv)
    same((V, X, lx, lv), want)
    P, V, X, W, (N, lx, lv) = fresh()
    nb.fwd_adjoint_step(p, P, V, W, X, W, lx, lv)
    same((V, W, lx, lv), want)
    P, V, X, W, (N, lx, lv) = fresh()
    nb.fwd_adjoint_step(p, P, V, N, X, W, P, lv)
    same((V, N, P, lv), want)
    for src in (2, 3):  # velocities in the storage of a cotangent
        t = fresh()
        nb.fwd_adjoint_step(p, t[0], t[src].clone(), t[4][0], t[2], t[3], *t[4][1:], cfg=two)
        want = t[4]
        t = fresh()
        nb.fwd_adjoint_step(p, t[0], t[src], t[4][0], t[2], t[3], *t[4][1:])
        same(t[4], want)

    P, V, X, W, (N, lx, lv) = fresh()
    v = P.clone()
    nb.forward_step(p, P, v, N, cfg=30)
    want = v, N
    P, V, X, W, (N, lx, lv) = fresh()
    nb.forward_step(p, P, P, N)
    same((P, N), want)
