"""What a user of this framework has it do, as cases that can be timed.

Every case goes through the plugin API (nbody_amd.HipBarnesHutNBodySimulation),
by `call`:

  frame      one GL_INTEROP step(): a Barnes-Hut step, then the vertices of all
             bodies on the host, as a renderer takes them for each picture
  run        `steps` steps of a simulation that goes on, then its vertices (a
             snapshot of a production run)
  restart    a simulation from given initial conditions: upload, `steps` steps,
             the state read back
  accel      accelerations of given bodies: upload, one force evaluation, read
             back (the engine as a force solver; nothing is advanced)
  train      the learned correction trained on a simulation's own pairs: the
             installed network and the report
  gradient   loss and gradient of the network on a batch of given pairs (the
             FP32 forward and backward passes)
  diagnose   energies, momenta and centre of mass, and the FP64 direct sum on
             sampled bodies (the accuracy yardstick)

A case's other fields are the universe (nbody_amd.universe), the number of
bodies and the simulation's parameters. Host arrays go in and come out: the
simulation keeps its bodies on the GPU behind its handle.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-nbody_amd"))

from nbody_amd import HipBarnesHutNBodySimulation, Mode, _lib, universe  # noqa: E402

# the reference's shipped constants: THETA 1.5 = theta^2, EPSILON 0.0025 =
# softening^2, TIMESTEP 0.025, work-group vote of 16 (the engine's defaults)
SHIPPED = dict(theta=math.sqrt(1.5), softening=0.05, dt=0.025, vote=16)
# of the larger runs: FP64 leapfrog positions, the update fused into the force
PRODUCTION = dict(softening=0.01, dt=1e-3, vote=64, fp64=True, fused=True)
LEARNED = dict(method="learned", coarse_theta=0.99, coarse_alpha=0.0175)

GENERATORS = {
    "rotating_disk": lambda n, seed: universe.rotating_disk(n, 3.5, 1.0, 1.0, seed=seed),
    "plummer_henon": lambda n, seed: universe.plummer_henon(n, seed=seed),
    "random_cubic": lambda n, seed: universe.random_cubic(n, 10.0, seed=seed),
    "uniform_ball": lambda n, seed: universe.uniform_ball(n, seed=seed),
    "plummer": lambda n, seed: universe.plummer(n, seed=seed),
    "two_plummer": lambda n, seed: universe.two_plummer(n, seed=seed),
    "gaussian_clusters": lambda n, seed: universe.gaussian_clusters(n, seed=seed),
    "halo_disk": lambda n, seed: universe.halo_disk(n, seed=seed),
}


def listed():
    return [
        # a small scene in the visualizer, at the reference's shipped constants:
        # the smallest call, all latency
        dict(name="frame 1000 disk", call="frame", universe="rotating_disk", n=1000, **SHIPPED),
        # the visualizer's own default universe (2048 * 16 bodies)
        dict(name="frame 32768 disk", call="frame", universe="rotating_disk", n=32768, **SHIPPED),
        # a short run from initial conditions: 16,384 bodies in a rotating ball,
        # ten steps, at the reference's vote width
        dict(name="restart 16384 ball vote 16", call="restart", universe="uniform_ball", n=16384, steps=10,
             theta=0.5, softening=0.05, dt=1e-3, vote=16),
        # a large scene at the engine's defaults, as a user gets who sets nothing;
        # a ragged number of bodies
        dict(name="run 1000003 shipped", call="run", universe="plummer_henon", n=1_000_003, steps=10, **SHIPPED),
        # an equilibrium Plummer sphere of 1M bodies in FP32, separate integrate
        dict(name="run 1M plummer", call="run", universe="plummer", n=1_048_576, steps=10, theta=0.5, softening=0.01,
             dt=1e-3, vote=64),
        # the benchmark universe, 4M clustered bodies: plain Barnes-Hut
        dict(name="run 4M clusters plain", call="run", universe="gaussian_clusters", n=4_194_304, steps=10, theta=0.4,
             **PRODUCTION),
        # the same with the learned coarse-theta force and its sampled FP64 check
        # every ten steps
        dict(name="run 4M clusters learned", call="run", universe="gaussian_clusters", n=4_194_304, steps=10,
             theta=0.4, **PRODUCTION, **LEARNED, check_every=10),
        # a halo and a disk under the coarse traversal without the network
        dict(name="run 700001 halo coarse", call="run", universe="halo_disk", n=700_001, steps=10, theta=0.4,
             **PRODUCTION, method="coarse", coarse_theta=0.8, coarse_alpha=0.02),
        # a force solver called with new bodies each time
        dict(name="accel 100003 two spheres", call="accel", universe="two_plummer", n=100_003, theta=0.4,
             softening=0.01, dt=1e-3, vote=64),
        # a network trained for a mid-sized run (a tenth of the default
        # iterations, at the default batch)
        dict(name="train 262144 clusters", call="train", universe="gaussian_clusters", n=262_144, steps=10,
             groups=256, iters=400, batch=4096, theta=0.4, **PRODUCTION, **LEARNED),
        # one gradient on a batch of the default size
        dict(name="gradient 4096 pairs", call="gradient", n=2048, rows=4096),
        # energy conservation and force error of a mid-sized run
        dict(name="diagnose 131072 halo", call="diagnose", universe="halo_disk", n=131_072, samples=1024, theta=0.4,
             **PRODUCTION),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["frame", "run", "run", "run", "restart", "accel", "train", "gradient", "diagnose"])
    if call == "frame":
        return dict(call=call, universe=rng.choice(["rotating_disk", "plummer_henon", "random_cubic"]),
                    n=_log_uniform(rng, 500, 65_536), **SHIPPED)
    if call == "run":
        kind = rng.choice(["shipped", "plain", "coarse", "learned"])
        n = _log_uniform(rng, 50_000, 1_500_000)
        if kind == "shipped":
            return dict(call=call, universe=rng.choice(["rotating_disk", "plummer_henon", "random_cubic"]), n=n,
                        steps=rng.randint(3, 10), **SHIPPED)
        case = dict(call=call, universe=rng.choice(["plummer", "two_plummer", "gaussian_clusters", "halo_disk"]), n=n,
                    steps=rng.randint(3, 10), **PRODUCTION)
        if kind == "plain":
            vote = rng.choice([16, 32, 64])
            return {**case, "theta": rng.choice([0.4, 0.5, 0.6]), "vote": vote, "fp64": rng.random() < 0.5,
                    "fused": rng.random() < 0.5}
        case = {**case, "theta": 0.4, "coarse_theta": rng.choice([0.8, 0.9, 0.99]),
                "coarse_alpha": rng.choice([0.0125, 0.0175, 0.025]), "method": kind}
        return {**case, "check_every": 10} if kind == "learned" else case
    if call == "restart":
        return dict(call=call, universe=rng.choice(["uniform_ball", "plummer"]), n=_log_uniform(rng, 2000, 200_000),
                    steps=rng.randint(5, 20), theta=rng.choice([0.5, 0.8]), softening=0.05, dt=1e-3,
                    vote=rng.choice([16, 32, 64]))
    if call == "accel":
        return dict(call=call, universe=rng.choice(["two_plummer", "gaussian_clusters", "halo_disk"]),
                    n=_log_uniform(rng, 5000, 500_000), theta=rng.choice([0.3, 0.4, 0.6]), softening=0.01, dt=1e-3,
                    vote=rng.choice([16, 64]))
    if call == "train":
        return dict(call=call, universe=rng.choice(["gaussian_clusters", "halo_disk"]),
                    n=_log_uniform(rng, 65_536, 1_000_000), steps=rng.randint(4, 10),
                    groups=rng.choice([128, 256, 512]), iters=rng.randint(100, 400),
                    batch=rng.choice([1000, 2048, 4096]), theta=0.4, **PRODUCTION, **LEARNED)
    if call == "gradient":
        return dict(call=call, n=2048, rows=_log_uniform(rng, 256, 65_536))
    return dict(call=call, universe=rng.choice(["plummer", "halo_disk"]), n=_log_uniform(rng, 10_000, 131_072),
                samples=rng.choice([512, 1024, 4096]), theta=0.4, **PRODUCTION)


def _universe(case, seed):
    return GENERATORS[case["universe"]](case["n"], int(seed) + 1)


def _model(seed):
    """A seeded network whose corrections are about 2e-4 of the acceleration,
    with feature scalings of the size that training finds."""
    g = universe.rng(seed)
    u = lambda shape, fan_in: g.uniform(-1.0, 1.0, shape) / math.sqrt(fan_in)
    weights = [u(24 * 64, 24), u(64, 24), u(64 * 64, 64), u(64, 64), u(64 * 3, 64), u(3, 64)]
    mean = [0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 6.2, 4.7, -3, -1.5, 0.95, -4, 0.3]
    sd = [0.3] * 3 + [0.1] * 2 + [0.2] * 3 + [0.5] * 3 + [0.3] * 3 + [0.1] * 3 + [0.3, 0.4, 1, 1, 0.05, 1, 0.5]
    return np.concatenate(weights + [mean, sd, np.zeros(3), np.full(3, 2e-4)]).astype(np.float32)


def _pairs(case, seed):
    g = universe.rng(int(seed) + 1)
    x = np.clip(g.normal(size=(case["rows"], 24)), -8, 8).astype(np.float32)
    t = np.clip(g.normal(size=(case["rows"], 3)), -8, 8).astype(np.float32)
    return x, t


def _simulation(case, state):
    flags = (_lib.NB_FP64_POSITIONS if case.get("fp64") else 0) | (_lib.NB_FUSED_UPDATE if case.get("fused") else 0)
    kw = dict(theta=case["theta"], softening=case["softening"], dt=case["dt"], vote_width=case["vote"], flags=flags)
    method = case.get("method", "plain")
    if method != "plain":
        kw.update(method=_lib.NB_MODE_LEARNED if method == "learned" else _lib.NB_MODE_COARSE,
                  coarse_theta=case["coarse_theta"], coarse_alpha=case["coarse_alpha"])
    if case.get("check_every"):
        # a tolerance that the traversal keeps: the check is paid for, the force stays learned
        kw.update(check_every=case["check_every"], check_samples=1024, check_tol=5e-3, check_adapt=1)
    mode = Mode.GL_INTEROP if case["call"] == "frame" else Mode.DEFAULT
    sim = HipBarnesHutNBodySimulation(mode, len(state[0]), universe.ArrayUniverse(state), **kw)
    sim.init(None)
    return sim


def prepare(case, seed):
    call = case["call"]
    if call == "gradient":
        state = universe.uniform_ball(case["n"], seed=int(seed) + 1)
        sim = _simulation(dict(call=call, theta=0.4, softening=0.01, dt=1e-3, vote=64, **LEARNED), state)
        sim.set_model(_model(int(seed) + 2))
        return dict(case=case, sim=sim, pairs=_pairs(case, seed))
    state = _universe(case, seed)
    sim = _simulation(case, state)
    held = dict(case=case, sim=sim)
    if call == "frame":
        sim.initGLBuffers(None, -1, -1)
    elif call == "run":
        if case.get("method") == "learned":
            # a learned run begins after the plain steps that its training pairs
            # came from: two of them here, then the network that the program keeps
            sim.train(steps=2, groups_per_step=16, iters=0, batch=64, seed=1)
            sim.set_model(_model(int(seed) + 2))
        held["vertices"] = [np.zeros((case["n"], 4), np.float32) for _ in range(2)]
    elif call in ("restart", "accel"):
        held["state"] = state
    elif call == "diagnose":
        held["sampled"] = _sampled(case, seed)
    return held


def _sampled(case, seed):
    return universe.rng(int(seed) + 3).permutation(case["n"])[:min(case["samples"], case["n"])].astype(np.int32)


def run(state):
    case, sim = state["case"], state["sim"]
    call = case["call"]
    if call == "frame":
        sim.step()
        return [sim.positions, sim.velocities]
    if call == "run":
        sim.steps(case["steps"])
        sim.copy_vertices(*state["vertices"])
        return state["vertices"]
    if call == "restart":
        sim.set_state(*state["state"])
        sim.steps(case["steps"])
        return sim.state()
    if call == "accel":
        sim.set_state(*state["state"])
        return sim.probe_accel()
    if call == "train":
        report = sim.train(steps=case["steps"], groups_per_step=case["groups"], iters=case["iters"],
                           batch=case["batch"], seed=1)
        return [sim.get_model(), report["samples"], report["loss_first"], report["loss_last"]]
    if call == "gradient":
        loss, grad = sim.mlp_loss_grad(*state["pairs"])
        return [loss, grad]
    d = sim.diagnostics()
    return [d["kinetic"], d["potential"], d["momentum"], d["angular_momentum"], d["centre_of_mass"], d["mass"],
            sim.direct_accel(state["sampled"])]


def _interactions(case):
    """About how many nodes a body meets under the opening test (per decade of
    bodies, as the angle sets it); the exact number depends on the positions."""
    n = case["n"]
    if case.get("method", "plain") == "plain":
        return min(n, 30.0 * math.log2(n) / case["theta"] ** 2)
    return min(n, 30.0 * math.log2(n))


def work(case):
    """20 operations per interaction (GPU Gems 3, chapter 31); each body's
    position, mass, velocity and acceleration read and written once a step,
    the pass's inputs and outputs moved once."""
    call, n = case["call"], case["n"]
    if call == "gradient":
        return dict(bytes=4.0 * (case["rows"] * 27 + 2 * 5955), flops=6.0 * 5955 * case["rows"])
    if call == "diagnose":
        return dict(bytes=32.0 * n, flops=20.0 * n * (n + case["samples"]))
    if call == "train":
        pairs = case["steps"] * case["groups"] * 64
        return dict(bytes=96.0 * n * case["steps"] + 108.0 * pairs + 108.0 * case["iters"] * case["batch"],
                    flops=20.0 * n * case["steps"] * min(n, 30.0 * math.log2(n) / case["theta"] ** 2)
                    + 6.0 * 5955 * case["iters"] * case["batch"])
    steps = case.get("steps", 1)
    return dict(bytes=96.0 * n * steps + 60.0 * n, flops=20.0 * n * steps * _interactions(case))


# ---- the same in 64 bits, by direct summation --------------------------------

def _direct(pos, m, eps2, targets=None, potential=False):
    """Softened accelerations (G = 1) at `targets` (all bodies by default), and
    with `potential` sum_{j != i} m_j / sqrt(r^2 + eps^2)."""
    who = torch.arange(len(pos), device=pos.device) if targets is None else targets
    out, phi = torch.empty(len(who), 3, dtype=torch.float64, device=pos.device), []
    block = max(1, 64_000_000 // len(pos))
    for i in range(0, len(who), block):
        w = who[i:i + block]
        r = [pos[None, :, k] - pos[w, k][:, None] for k in range(3)]
        inv = (r[0] * r[0] + r[1] * r[1] + r[2] * r[2] + eps2).rsqrt_()
        if potential:
            phi.append(inv @ m - m[w] / math.sqrt(eps2))
        f = inv.pow_(3).mul_(m[None, :])
        for k in range(3):
            out[i:i + block, k] = (f * r[k]).sum(1)
    return (out, torch.cat(phi)) if potential else out


def _on_gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", torch.float64)


def exact(case, seed):
    """Direct sums where the engine approximates by its tree, so the distance
    includes the tree's own error (the same before and after a change)."""
    call, n = case["call"], case["n"]
    if call == "gradient":
        x, t = (_on_gpu(a) for a in _pairs(case, seed))
        flat = _on_gpu(_model(int(seed) + 2)[:5955]).requires_grad_()
        w1, b1, w2, b2, w3, b3 = torch.split(flat, [24 * 64, 64, 64 * 64, 64, 64 * 3, 3])
        gelu = lambda v: torch.nn.functional.gelu(v, approximate="tanh")
        h = gelu(gelu(x @ w1.view(24, 64) + b1) @ w2.view(64, 64) + b2)
        loss = ((h @ w3.view(64, 3) + b3 - t) ** 2).mean()
        loss.backward()
        return [loss.detach(), flat.grad]
    if call in ("run", "train") or n > 200_000:
        return None
    st = _universe(case, seed)
    pos, vel = (torch.stack([_on_gpu(a) for a in st[k:k + 3]], 1) for k in (0, 3))
    m = _on_gpu(st[6])
    # the engine squares the softening and steps in FP32 constants
    eps2, dt = float(np.float32(case["softening"]) * np.float32(case["softening"])), float(np.float32(case["dt"]))
    if call == "accel":
        return _direct(pos, m, eps2)
    if call == "diagnose":
        _, phi = _direct(pos, m, eps2, potential=True)
        mass = m.sum()
        return [0.5 * (m * (vel * vel).sum(1)).sum(), -0.5 * (m * phi).sum(), (m[:, None] * vel).sum(0),
                (m[:, None] * torch.linalg.cross(pos, vel)).sum(0), (m[:, None] * pos).sum(0) / mass, mass,
                _direct(pos, m, eps2, torch.from_numpy(_sampled(case, seed).astype(np.int64)).cuda())]
    if n > 70_000:
        return None
    old = None
    for _ in range(case.get("steps", 1)):
        a = _direct(pos, m, eps2)
        if old is not None:
            vel = vel + (a - old) * (0.5 * dt)
        old = a
        half = vel + a * (0.5 * dt)
        pos = pos + half * dt
        vel = half + a * (0.5 * dt)
    if call == "frame":
        one = torch.ones(n, 1, dtype=torch.float64, device=pos.device)
        return [torch.cat([pos, one], 1), torch.cat([vel, one], 1)]
    return [pos[:, 0], pos[:, 1], pos[:, 2], vel[:, 0], vel[:, 1], vel[:, 2]]
