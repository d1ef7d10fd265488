"""A stream's scratch, sized by one step, serves captured steps of other rules on
the same particles and captured diagnostics."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(nb, gpu, n):
    import torch

    pos, vel = nb.plummer_ic(n, seed=n, g_mass=1.0)
    P, V = (torch.from_numpy(np.stack(a)).to(gpu) for a in (pos, vel))
    gen = torch.Generator().manual_seed(n)
    lam = [torch.randn(3, n, generator=gen).to(gpu) for _ in range(2)]
    return nb.default_params(num_particles=n, G=1.0 / n), P, V, *lam


def _call(nb, kind, p, P, V, lxn, lvn, stream):
    import torch

    v, a, b, c = V.clone(), *(torch.empty_like(P) for _ in range(3))
    if kind == "plain" or kind == "kahan":
        nb.forward_step(p, P, v, a, acc=int(kind == "kahan"), stream=stream)
    elif kind == "adjoint":
        nb.adjoint_step(p, P, lxn, lvn, b, c, stream=stream)
    elif kind == "fused":
        nb.fwd_adjoint_step(p, P, v, a, lxn, lvn, b, c, stream=stream)
    else:
        idx = torch.arange(0, P.shape[1], 3, dtype=torch.int32, device=P.device)
        return [nb.forces_f64(p, P, idx, stream=stream)]
    return {"plain": [v, a], "kahan": [v, a], "adjoint": [b, c], "fused": [v, a, b, c]}[kind]


@pytest.mark.parametrize("n, warm, kinds", [
    (1000, "plain", ["forces"]), (1000, "kahan", ["forces"]), (2000, "adjoint", ["forces"]),
    (4096, "plain", ["kahan", "fused", "forces"]), (9000, "plain", ["kahan"]),
    (12287, "plain", ["kahan"]), (12287, "forces", ["kahan"]),
    (20480, "plain", ["fused", "adjoint"]), (32767, "plain", ["fused"])])
def test_captured_after_another_call(nb, gpu, n, warm, kinds):
    import torch

    st = _state(nb, gpu, n)
    want = {k: _call(nb, k, *st, torch.cuda.current_stream()) for k in kinds}
    torch.cuda.synchronize()
    nb.scratch_release()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        _call(nb, warm, *st, s)
    s.synchronize()
    for k in kinds:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            got = _call(nb, k, *st, s)
        for _ in range(3):
            for t in got:
                t.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want[k])), k


def test_first_small_step_beside_a_capture(nb, gpu):
    """A one-launch step on a stream without a buffer, while another stream is
    being captured, runs and leaves the capture whole."""
    import torch

    st = _state(nb, gpu, 1000)
    want = _call(nb, "plain", *st, torch.cuda.current_stream())
    torch.cuda.synchronize()
    nb.scratch_release()
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    p, P, V = st[:3]
    v, N, cv, cN = V.clone(), torch.empty_like(P), V.clone(), torch.empty_like(P)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        nb.forward_step(p, P, cv, cN, stream=s)
        nb.forward_step(p, P, v, N, stream=other)
    torch.cuda.synchronize()
    assert torch.equal(v, want[0]) and torch.equal(N, want[1])
    for _ in range(3):
        cv.copy_(V)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(cv, want[0]) and torch.equal(cN, want[1])
