"""The ways of the build by size: one block or many for the bounding box (up to
32,768 bodies and past it), the scan of the bucket counts inside the scatter (up
to 1023 splitters of 256 bodies: 261,888 bodies) or before it, and the cells
grouped by level inside the build (up to 524,288 bodies) or after it. At each
edge a first build and a warm one, stage by stage and out of step (a build
without a new bounding box), against the oracle: paths, depths, order and cell
counts are integers and equal.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim

pytestmark = pytest.mark.gpu


def _same_tree(sim, orc, n):
    assert orc.run_stages(1, 2) == 0
    gp, gd = sim.paths()
    op, od = orc.paths()
    assert np.array_equal(gd, od)
    assert np.array_equal(gp, op)
    for stage in (3, 4):
        sim.run_stage(stage)
    assert orc.run_stages(3, 4) == 0
    assert np.array_equal(sim.sorted(), orc.sorted())
    g, o = np.sort(sim.cells()["count"]), np.sort(orc.cells()["count"])
    assert np.array_equal(g, o) and g[-1] == n


@pytest.mark.parametrize("n", [1, 2, 513, 1025, 32_768, 32_769, 261_888, 261_889, 524_288, 524_289])
def test_build_at_size_edges(nb, oracle, n):
    from nbody_amd import universe as U

    st = U.plummer_henon(n, seed=5 + n % 89)
    kw = dict(theta=1.2, softening=0.05, dt=5e-3)
    sim = make_sim(st, vote_width=64, **kw)
    for repeat in (1, 2):  # from scratch, then from the order of the last tree
        for stage in (1, 2):
            sim.run_stage(stage)
        x, y, z, vx, vy, vz = sim.state()
        orc = make_oracle((x, y, z, vx, vy, vz, st[6]), kw["theta"], kw["softening"], kw["dt"], 64)
        _same_tree(sim, orc, n)
        sim.run_stage(2)  # the same box, now from this tree's order
        orc = make_oracle((x, y, z, vx, vy, vz, st[6]), kw["theta"], kw["softening"], kw["dt"], 64)
        _same_tree(sim, orc, n)
        sim.steps(1)
    sim.close()
