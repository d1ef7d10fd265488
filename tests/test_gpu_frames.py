"""Frames on both sides of the line between direct launches and graph replay
advance the same states, also when their lengths change from frame to frame."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 700, 4095, 4097])
@pytest.mark.parametrize("acc", [0, 1])
def test_mixed_frames(nb, gpu, n, acc):
    frames = [5, 6, 2, 3, 6, 1, 6, 3, 5, 7]
    pos, vel = nb.plummer_ic(n, seed=2, g_mass=1.0)
    out = []
    for graph in (True, False):
        p = nb.default_params(num_particles=n, G=1.0 / n, dist_eps=1e-2)
        s = nb.Simulator(p, pos, vel)
        s.set_accumulation(acc)
        s.set_graph(graph)
        states = []
        for f in frames:
            s.set_frame_iterations(f)
            s.step_sim()
            states.append(np.stack([*s.positions(), *s.velocities()]))
        out.append(states)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
