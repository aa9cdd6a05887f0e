"""Steps whose force pass only stores accelerations, followed by the integrate
kernel: with timing on and NB_FUSED_UPDATE off every stage is a launch of its own
(steps in one call advance the bodies in the force pass in any case). The next
build then gathers the records instead of reading them in the last order.

Against the oracle on the universes of the parity tests, and against whole steps,
bit for bit, in coarse and learned mode on both sides of every number of waves
per group. Such steps in plain mode are compared in test_gpu_whole_steps.py.
"""
import numpy as np
import pytest

from helpers import cell_multiset, make_oracle, make_sim, random_model
from test_gpu_parity import PHYS, _collapse, _universes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,dt,large", [("plummer_32k", 0.0, False), ("plummer_32k", 1e-3, False),
                                           ("tight_run_8219", 1e-3, False), ("collapse_32k", 1.0, True)])
def test_warm_build_from_gathered_records(nb, oracle, case, dt, large):
    st = _collapse() if case == "collapse_32k" else _universes()[case]()
    sim = make_sim(st, theta=0.5, softening=0.05, dt=dt)
    sim.set_timing(True)
    sim.steps(1)
    x, y, z, vx, vy, vz = sim.state()
    orc = make_oracle((x, y, z, vx, vy, vz, st[6]), 0.5, 0.05, dt, 16)
    before = sim.counters().large_buckets
    for stage in range(1, 5):
        sim.run_stage(stage)
    assert orc.run_stages(1, 2) == 0
    gp, gd = sim.paths()
    op, od = orc.paths()
    assert np.array_equal(gd, od) and gd.min() > 0 and np.array_equal(gp, op)
    assert orc.run_stages(3, 4) == 0
    gc, oc = sim.cells(), orc.cells()
    assert np.array_equal(cell_multiset(gc["count"], gc["x"], gc["y"], gc["z"], gc["m"]),
                          cell_multiset(oc["count"], oc["x"], oc["y"], oc["z"], oc["m"]))
    assert np.array_equal(sim.sorted(), orc.sorted())
    assert (sim.counters().large_buckets > before) == large
    sim.close()


def test_steps_track_oracle(nb, oracle):
    st = _universes()["uniform_ball_16k"]()
    sim = make_sim(st, **PHYS)
    sim.set_timing(True)
    orc = make_oracle(st, 0.5, 0.05, 1e-3, 16)
    for k in range(3):
        acc = sim.accel()
        orc.set_state(*sim.state(), st[6])
        orc.set_accel(acc[:, 0], acc[:, 1], acc[:, 2], k - 1)
        sim.steps(1)
        assert orc.step(1) == 0
        g, o = (np.stack(s.state(), axis=1) for s in (sim, orc))
        d = np.abs(g.astype(np.float64) - o) / np.maximum(np.abs(o), 1e-3)
        assert d.max() < 1e-6, (k, d.max())
    sim.close()


def test_single_body(nb, oracle):
    st = tuple(np.array([v], np.float32) for v in (0.25, -0.5, 1.0, 0.3, -0.2, 0.1, 2.0))
    sim = make_sim(st, **PHYS)
    sim.set_timing(True)
    orc = make_oracle(st, 0.5, 0.05, 1e-3, 16)
    sim.steps(3)
    assert orc.step(3) == 0
    g, o = (np.array(s.state(), np.float32) for s in (sim, orc))
    assert np.array_equal(g.view(np.uint32), o.view(np.uint32))
    sim.close()


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("method", ["coarse", "learned"])
@pytest.mark.parametrize("n", [1000, 20_481, 81_921, 589_825])
def test_whole_steps_equal_stages(nb, n, method, fp64):
    from nbody_amd import _lib, universe as U

    st = U.gaussian_clusters(n, seed=n % 31)
    sims = []
    for flags, timing in ((0, False), (0, True), (_lib.NB_FUSED_UPDATE, True)):
        sim = make_sim(st, theta=0.4, softening=0.01, dt=1e-3, vote_width=64, coarse_theta=0.9, coarse_alpha=0.02,
                       method=_lib.NB_MODE_LEARNED if method == "learned" else _lib.NB_MODE_COARSE,
                       flags=flags | (_lib.NB_FP64_POSITIONS if fp64 else 0))
        if method == "learned":
            sim.set_model(random_model(3))
        sim.set_timing(timing)
        sim.steps(2)
        sim.steps(1)
        sims.append((sim.state(), sim.accel(), sim.sorted()))
        sim.close()
    for state, acc, order in sims[1:]:
        for a, b in zip(state, sims[0][0]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert np.array_equal(acc, sims[0][1]) and np.array_equal(order, sims[0][2])
