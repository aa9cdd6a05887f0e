"""Stages run one by one in another order than a step's: a summarize after a
bounding box and no build finds the root alone, without bodies (the box turns
every child slot stale), whether the build groups the cells by level itself (up to
524,288 bodies) or not. The next build starts over."""
import numpy as np
import pytest

from helpers import make_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vote", [16, 64])
@pytest.mark.parametrize("n", [1000, 60_000, 524_289])
def test_summarize_without_a_build(nb, n, vote):
    from nbody_amd import universe as U

    sim = make_sim(U.plummer(n, seed=3), theta=0.8, softening=0.05, dt=1e-3, vote_width=vote)
    for stage in range(1, 6):
        sim.run_stage(stage)
    acc = sim.accel()
    assert np.linalg.norm(acc, axis=1).min() > 0
    cells = sim.counters().live_cells
    for stage in (1, 3):
        sim.run_stage(stage)
    assert sim.counters().live_cells == 1 and list(sim.cells()["count"]) == [0]
    for stage in range(1, 6):
        sim.run_stage(stage)
    assert sim.counters().live_cells == cells and np.array_equal(sim.accel(), acc)
    sim.close()
