"""The work a user of nbody_amd has it do, as measurable cases.

Each case is one call (or one short sequence of calls) through the package's
public entry points on inputs made from a seed:

  step         forward_step: one all-pairs step on device tensors, plain or
               Kahan sums;
  frame        Simulator.step_sim + staged: a driver's frame (SimParam's four
               iterations per frame) and the readback of its particles;
  adjoint      adjoint_step: one reverse step on device tensors;
  fused        fwd_adjoint_step: the forward and the reverse step together;
  trajectory   trajectory + backward: a checkpointed differentiable run;
  batch        Batch.step: many independent systems, autotuned, then read back;
  diagnostics  energy_momentum and forces_f64: the fp64 checks of a state.

Initial conditions: "disk" is the reference's generator (positions up to 100,
a few very close pairs), "plummer" a virial sphere of unit total mass.  The
disk is chaotic over several steps (its close pairs at eps = 1e-7 amplify a
rounding a thousandfold within four steps), so the multi-step cases run the
Plummer sphere, or the disk with the softening of the conditioned trajectory
tests (1e-2).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "cuda-to-sycl-nbody_amd"))

import nbody_amd as nb  # noqa: E402

_MAX_STEP = 262144     # the headline size
_MAX_HEAVY = 200000    # Kahan sums and adjoint steps cost 1.7 to 2.2 plain ones


def listed():
    return [
        # a small system stepped from a user's loop: launches are the cost
        {"name": "step_1000", "kind": "step", "n": 1000, "ic": "plummer", "acc": "plain"},
        # a few thousand particles, one past a power of two
        {"name": "step_4097", "kind": "step", "n": 4097, "ic": "disk", "acc": "plain"},
        # SimParam's default particle count (50 x 256)
        {"name": "step_12800", "kind": "step", "n": 12800, "ic": "disk", "acc": "plain"},
        # a mid-sized, odd particle count
        {"name": "step_50021", "kind": "step", "n": 50021, "ic": "disk", "acc": "plain"},
        # the headline benchmark (1024 x 256)
        {"name": "step_262144", "kind": "step", "n": 262144, "ic": "disk", "acc": "plain"},
        # a precision-minded run: compensated force sums
        {"name": "kahan_30001", "kind": "step", "n": 30001, "ic": "disk", "acc": "kahan"},
        # one frame of the driver's loop with its readback, default size
        {"name": "frame_12800", "kind": "frame", "n": 12800, "iterations": 4},
        # one reverse step at the trajectory workload's size
        {"name": "adjoint_16384", "kind": "adjoint", "n": 16384},
        # forward and reverse step together, large and odd
        {"name": "fused_100003", "kind": "fused", "n": 100003},
        # gradient through 20 steps, a checkpoint every 10, at the trajectory workload's size
        {"name": "trajectory_16384", "kind": "trajectory", "n": 16384, "steps": 20, "every": 10},
        # the batched benchmark's 64 uneven systems (1024 to 32768 particles)
        {"name": "batch_64", "kind": "batch", "systems": 64, "lo": 1024, "hi": 32768,
         "sizes_seed": 0, "steps": 4},
        # a state's energy, momentum and 4096 sampled fp64 forces
        {"name": "diagnostics_65536", "kind": "diagnostics", "n": 65536, "samples": 4096},
    ]


def _size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, n))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "kahan", "kahan", "frame", "adjoint",
                       "adjoint", "fused", "fused", "trajectory", "batch", "diagnostics"])
    if kind == "step":
        return {"kind": "step", "n": _size(rng, 200, _MAX_STEP),
                "ic": rng.choice(["disk", "plummer"]), "acc": "plain"}
    if kind == "kahan":
        return {"kind": "step", "n": _size(rng, 500, _MAX_HEAVY),
                "ic": rng.choice(["disk", "plummer"]), "acc": "kahan"}
    if kind == "frame":
        return {"kind": "frame", "n": _size(rng, 500, 50000), "iterations": rng.randint(1, 8)}
    if kind == "adjoint":
        return {"kind": "adjoint", "n": _size(rng, 500, _MAX_HEAVY)}
    if kind == "fused":
        return {"kind": "fused", "n": _size(rng, 500, _MAX_HEAVY)}
    if kind == "trajectory":
        return {"kind": "trajectory", "n": _size(rng, 1000, 16384), "steps": rng.randint(5, 20),
                "every": rng.choice([5, 10])}
    if kind == "batch":
        return {"kind": "batch", "systems": rng.randint(4, 64), "lo": rng.choice([256, 512, 1024]),
                "hi": 256 * rng.randint(16, 128), "sizes_seed": rng.randint(0, 999),
                "steps": rng.randint(1, 4)}
    return {"kind": "diagnostics", "n": _size(rng, 1000, 65536), "samples": rng.randint(100, 4096)}


# ---- inputs -----------------------------------------------------------------


def _ics(ic, n, seed):
    """Host arrays ((x, y, z), (vx, vy, vz)) and the parameters they go with."""
    if ic == "plummer":
        pos, vel = nb.plummer_ic(n, seed=seed % (1 << 31), a=1.0, g_mass=1.0)
        return pos, vel, nb.default_params(num_particles=n, G=1.0 / n)
    pos, vel = nb.disk_ic(n, seed=seed % (1 << 31))
    return pos, vel, nb.default_params(num_particles=n)


def _dev(rows):
    return torch.from_numpy(np.stack(rows)).cuda()


def _cotangents(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(3, n, generator=g, device="cuda"),
            torch.randn(3, n, generator=g, device="cuda"))


def _batch_inputs(case, seed):
    """Uneven Plummer systems, back to back, as the batched benchmark makes them."""
    sizes = nb.plummer_batch_sizes(case["systems"], seed=case["sizes_seed"], lo=case["lo"],
                                   hi=case["hi"])
    params, pos, vel = [], [[], [], []], [[], [], []]
    for k, m in enumerate(sizes):
        p, v, par = _ics("plummer", m, seed + 1 + k)
        params.append(par)
        for c in range(3):
            pos[c].append(p[c])
            vel[c].append(v[c])
    return (sizes, params, tuple(np.concatenate(a) for a in pos),
            tuple(np.concatenate(a) for a in vel))


def _samples(case, seed):
    g = torch.Generator().manual_seed(seed)
    m = min(case["samples"], case["n"])
    return torch.sort(torch.randperm(case["n"], generator=g)[:m])[0].to(torch.int32).cuda()


def _trajectory_params(n):
    return nb.default_params(num_particles=n, dist_eps=1e-2)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "batch":
        # a user creates the batch once and lets it pick its launch shape
        _, params, pos, vel = _batch_inputs(case, seed)
        s["batch"] = nb.Batch(params, pos, vel)
        s["batch"].autotune(2)
        return s
    n = case["n"]
    if kind == "frame":
        pos, vel, params = _ics("plummer", n, seed)
        params.sim_iterations_per_frame = case["iterations"]
        s["sim"] = nb.Simulator(params, pos, vel)
        return s
    pos, vel, params = _ics(case.get("ic", "disk"), n, seed)
    s["params"] = params
    s["pos"], s["vel"] = _dev(pos), _dev(vel)
    if kind == "step":
        s["nxt"] = torch.empty_like(s["pos"])
        s["acc"] = nb.NB_ACC_KAHAN if case["acc"] == "kahan" else nb.NB_ACC_PLAIN
    elif kind in ("adjoint", "fused"):
        s["nxt"] = torch.empty_like(s["pos"])
        s["lxn"], s["lvn"] = _cotangents(n, seed)
        s["lx"], s["lv"] = torch.empty_like(s["lxn"]), torch.empty_like(s["lvn"])
    elif kind == "trajectory":
        s["params"] = _trajectory_params(n)
        s["target"] = s["pos"] + 10.0
        s["pos"].requires_grad_(True)
        s["vel"].requires_grad_(True)
    elif kind == "diagnostics":
        s["idx"] = _samples(case, seed)
    return s


# ---- one pass -----------------------------------------------------------------


def run(s):
    kind = s["kind"]
    if kind == "step":
        nb.forward_step(s["params"], s["pos"], s["vel"], s["nxt"], acc=s["acc"])
        return {"next": s["nxt"], "vel": s["vel"]}
    if kind == "frame":
        s["sim"].step_sim()
        pos, vel = s["sim"].staged()
        return {"pos": list(pos), "vel": list(vel)}
    if kind == "adjoint":
        nb.adjoint_step(s["params"], s["pos"], s["lxn"], s["lvn"], s["lx"], s["lv"])
        return {"lx": s["lx"], "lv": s["lv"]}
    if kind == "fused":
        nb.fwd_adjoint_step(s["params"], s["pos"], s["vel"], s["nxt"], s["lxn"], s["lvn"],
                            s["lx"], s["lv"])
        return {"next": s["nxt"], "vel": s["vel"], "lx": s["lx"], "lv": s["lv"]}
    if kind == "trajectory":
        x, v = s["pos"], s["vel"]
        x.grad = v.grad = None
        xT, vT = nb.trajectory(x, v, s["params"], s["case"]["steps"], s["case"]["every"])
        ((xT - s["target"]) ** 2).sum(0).mean().backward()
        return {"x": xT.detach(), "v": vT.detach(), "gx": x.grad, "gv": v.grad}
    if kind == "batch":
        s["batch"].step(s["case"]["steps"])
        return {"pos": list(s["batch"].positions()), "vel": list(s["batch"].velocities())}
    e = nb.energy_momentum(s["params"], s["pos"], s["vel"])
    return {"kinetic": e["kinetic"], "potential": e["potential"], "total": e["total"],
            "momentum": list(e["momentum"]),
            "forces": nb.forces_f64(s["params"], s["pos"], s["idx"])}


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    """Bytes: inputs read once, outputs written once.  Flops: each unordered
    pair's term once (fma = 2, rsqrt = 1): forward 24 (3 sub, |r|^2 + eps 6,
    d^3 2, rsqrt 1, both sums 12), adjoint 43, forward and adjoint 54, Kahan
    sums 18 more than plain."""
    kind = case["kind"]
    if kind == "batch":
        sizes = nb.plummer_batch_sizes(case["systems"], seed=case["sizes_seed"], lo=case["lo"],
                                       hi=case["hi"])
        n1, pairs = float(sum(sizes)), 0.5 * sum(m * (m - 1.0) for m in sizes)
        return {"bytes": 48.0 * n1 * case["steps"], "flops": 24.0 * pairs * case["steps"]}
    n = case["n"]
    pairs = 0.5 * n * (n - 1)
    if kind == "step":
        return {"bytes": 48.0 * n, "flops": (42.0 if case["acc"] == "kahan" else 24.0) * pairs}
    if kind == "frame":
        return {"bytes": 48.0 * n * case["iterations"], "flops": 24.0 * pairs * case["iterations"]}
    if kind == "adjoint":
        return {"bytes": 60.0 * n, "flops": 43.0 * pairs}
    if kind == "fused":
        return {"bytes": 96.0 * n, "flops": 54.0 * pairs}
    if kind == "trajectory":
        t = case["steps"]
        return {"bytes": (48.0 + 60.0) * n * t, "flops": (24.0 + 43.0) * pairs * t}
    m = min(case["samples"], n)
    return {"bytes": 24.0 * n + 28.0 * m, "flops": 14.0 * pairs + 22.0 * m * n}


# ---- 64-bit results -------------------------------------------------------------


def _f32(v):
    return float(np.float32(v))


def _rows(n):
    """Target rows per block: keeps a block's pair matrix at 2^25 doubles."""
    return max(1, min(n, (1 << 25) // max(n, 1)))


def _force64(x, eps, idx=None):
    """Sum over j of r K, K = (|r|^2 + eps)^-3/2 (the self term is zero: r = 0)."""
    t = x if idx is None else x[:, idx]
    out = torch.empty_like(t)
    step = _rows(x.shape[1])
    for i in range(0, t.shape[1], step):
        r = x[:, None, :] - t[:, i:i + step, None]
        d = r.square().sum(0) + eps
        k = 1.0 / (d * d.sqrt())
        out[:, i:i + step] = (r * k).sum(2)
    return out


def _adjoint64(x, g, eps):
    """Sum over j of K (h - 3 r (r . h) / d), h = g_j - g_k."""
    out = torch.empty_like(x)
    step = _rows(x.shape[1])
    for i in range(0, x.shape[1], step):
        r = x[:, None, :] - x[:, i:i + step, None]
        h = g[:, None, :] - g[:, i:i + step, None]
        d = r.square().sum(0) + eps
        k = 1.0 / (d * d.sqrt())
        t3 = -3.0 * (r * h).sum(0) / d
        out[:, i:i + step] = (k * (h + t3 * r)).sum(2)
    return out


def _step64(x, v, eps, damping, dt, G):
    v1 = damping * v + dt * G * _force64(x, eps)
    return x + dt * v1, v1


def _back64(x, lx, lv, eps, damping, dt, G):
    g = lv + dt * lx
    return lx + dt * G * _adjoint64(x, g, eps), damping * g


def _consts(p):
    return _f32(p.dist_eps), _f32(p.damping), _f32(p.dt), _f32(p.G)


def _state64(pos, vel):
    where = "cuda" if torch.cuda.is_available() else "cpu"
    return (torch.from_numpy(np.stack(pos)).to(where, torch.float64),
            torch.from_numpy(np.stack(vel)).to(where, torch.float64))


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        sizes, params, pos, vel = _batch_inputs(case, seed)
        X, V, o = [], [], 0
        for m, p in zip(sizes, params):
            x, v = _state64([a[o:o + m] for a in pos], [a[o:o + m] for a in vel])
            for _ in range(case["steps"]):
                x, v = _step64(x, v, *_consts(p))
            X.append(x)
            V.append(v)
            o += m
        return {"pos": list(torch.cat(X, 1)), "vel": list(torch.cat(V, 1))}
    n = case["n"]
    pos, vel, params = _ics("plummer" if kind == "frame" else case.get("ic", "disk"), n, seed)
    x, v = _state64(pos, vel)
    if kind == "trajectory":
        c = _consts(_trajectory_params(n))
        states = [x]
        target = (x.float() + 10.0).double()
        for _ in range(case["steps"]):
            x, v = _step64(x, v, *c)
            states.append(x)
        lx, lv = 2.0 * (x - target) / n, torch.zeros_like(x)
        for s in reversed(states[:-1]):
            lx, lv = _back64(s, lx, lv, *c)
        return {"x": x, "v": v, "gx": lx, "gv": lv}
    c = _consts(params)
    if kind == "diagnostics":
        w = 0.0
        for i in range(0, n, _rows(n)):
            r = x[:, None, :] - x[:, i:i + _rows(n), None]
            q = 1.0 / (r.square().sum(0) + c[0]).sqrt()
            w += float(q.sum()) - q.shape[0] / math.sqrt(c[0])
        k = 0.5 * float(v.square().sum())
        w = -0.5 * c[3] * w
        idx = _samples(case, seed).long().to(x.device)
        return {"kinetic": k, "potential": w, "total": k + w, "momentum": v.sum(1).tolist(),
                "forces": _force64(x, c[0], idx)}
    if kind == "frame":
        for _ in range(case["iterations"]):
            x, v = _step64(x, v, *c)
        return {"pos": list(x), "vel": list(v)}
    if kind == "step":
        x1, v1 = _step64(x, v, *c)
        return {"next": x1, "vel": v1}
    lxn, lvn = _cotangents(n, seed)
    lx, lv = _back64(x, lxn.double().to(x.device), lvn.double().to(x.device), *c)
    if kind == "adjoint":
        return {"lx": lx, "lv": lv}
    x1, v1 = _step64(x, v, *c)
    return {"next": x1, "vel": v1, "lx": lx, "lv": lv}
