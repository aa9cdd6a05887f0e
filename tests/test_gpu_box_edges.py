"""The bounding box on both sides of the size up to which one block works it out
(24,576 bodies): root bit for bit, and the splitters that go with it, by the order
of the warm build that uses them."""
import numpy as np
import pytest

from helpers import make_oracle, make_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 24_575, 24_576, 24_577, 24_833])
def test_box_at_one_block_edge(nb, oracle, n):
    from nbody_amd import universe as U

    st = U.uniform_ball(n, seed=n % 41)
    sim = make_sim(st, theta=0.8, softening=0.05, dt=0.02)
    for _ in range(2):  # the second box comes with splitters
        x, y, z, vx, vy, vz = sim.state()
        orc = make_oracle((x, y, z, vx, vy, vz, st[6]), 0.8, 0.05, 0.02, 16)
        for stage in range(1, 5):
            sim.run_stage(stage)
        assert orc.run_stages(1, 1) == 0  # before its summarize moves the root's record to the centre of mass
        assert np.array_equal(sim.root().view(np.uint32), orc.root().view(np.uint32))
        assert orc.run_stages(2, 4) == 0
        assert np.array_equal(sim.sorted(), orc.sorted())
        sim.steps(1)
    sim.close()
