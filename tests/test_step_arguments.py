"""Step tensors given as one (3, n) tensor and as three rows: the same results,
and the same arguments refused."""
import numpy as np
import pytest


def _forms(torch, t, n):
    """The same rows in every accepted form."""
    wide = torch.zeros(3, n + 7, device=t.device)
    wide[:, 2:n + 2] = t
    sub = torch.nn.Parameter(t.clone(), requires_grad=False)
    cols = torch.zeros(n, 3, device=t.device).t().contiguous()
    cols.copy_(t)
    return [t.clone(), [r.clone() for r in t], tuple(t.clone()), wide[:, 2:n + 2], sub, cols,
            torch.cat([t, t])[3:]]


def test_cpu_tensors_take_the_general_checks(nb):
    import torch

    from nbody_amd._rows import row_length, row_ptrs

    t = torch.zeros(3, 8)
    assert row_ptrs(t, 8) is None and row_length(t) == 8 and row_length(list(t)) == 8
    with pytest.raises(ValueError):
        nb.forward_step(nb.default_params(num_particles=8), t, t.clone(), t.clone())
    with pytest.raises(ValueError):
        nb.adjoint_step(nb.default_params(num_particles=8), *[t.clone() for _ in range(5)])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 33, 500])
def test_forms_agree(nb, gpu, n):
    import torch

    pos, vel = nb.disk_ic(n)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    p = nb.default_params(num_particles=n)
    out = []
    for pf, vf, nf in zip(_forms(torch, P, n), _forms(torch, V, n), _forms(torch, P * 0, n)):
        lx, lv = [r.clone() for r in P], [r.clone() for r in P]
        nb.adjoint_step(p, pf, vf, vf, lx, lv)
        nb.forward_step(p, pf, vf, nf)
        out.append(torch.stack([*vf, *nf, *lx, *lv]).cpu().numpy())
    for o in out[1:]:
        assert np.array_equal(o, out[0])


@pytest.mark.gpu
def test_refused_arguments(nb, gpu):
    import torch

    n = 64
    p = nb.default_params(num_particles=n)
    good = lambda: torch.randn(3, n, device=gpu)
    for bad in (torch.randn(n, 3, device=gpu).t(), torch.randn(3, 2 * n, device=gpu)[:, ::2],
                good().double(), good().cpu(), torch.randn(3, n - 1, device=gpu),
                torch.randn(4, n, device=gpu), torch.randn(2, n, device=gpu)):
        for k in (1, 2):
            a = [good(), good(), good()]
            a[k] = bad
            with pytest.raises(ValueError):
                nb.forward_step(p, *a)
        for k in range(1, 5):
            a = [good() for _ in range(5)]
            a[k] = bad
            with pytest.raises(ValueError):
                nb.adjoint_step(p, *a)


@pytest.mark.gpu
def test_current_stream_is_used(nb, gpu):
    import torch

    n = 400
    pos, vel = nb.disk_ic(n)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    p = nb.default_params(num_particles=n)
    N, v = torch.zeros_like(P), V.clone()
    nb.forward_step(p, P, v, N)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    g, gv, gn = torch.cuda.CUDAGraph(), V.clone(), torch.zeros_like(P)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):  # fails unless it is on `side`
        nb.forward_step(p, P, gv, gn)
    for _ in range(3):
        gv.copy_(V)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gn, N) and torch.equal(gv, v)
