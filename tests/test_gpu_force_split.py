"""The force traversal on both sides of every number of bodies at which the
number of waves per group changes (40,960, 114,688 and 327,680 bodies: 640, 1,792
and 5,120 groups of 64), with a last group that is full, holds one body, or ends
inside a vote group, at the three vote widths.

The oracle takes the same opening decisions, so the interaction counts are
equal; its sums are FP64 and the engine's FP32 terms carry a few roundings
each (1e-5 relative, the bar of the other parity tests). A probe repeats bit for
bit: the waves of a group share their work by an order that only the tree sets.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vote", [16, 32, 64])
@pytest.mark.parametrize("n", [1, 63, 40_960, 40_961, 114_688, 114_715, 327_680, 327_699])
def test_force_at_split_edges(nb, oracle, n, vote):
    from nbody_amd import universe as U

    st = U.plummer_henon(n, seed=n % 97 + vote)
    kw = dict(theta=1.2, softening=0.05, dt=1e-3)
    sim = make_sim(st, vote_width=vote, **kw)
    for s in range(1, 6):
        sim.run_stage(s)
    orc = make_oracle(st, kw["theta"], kw["softening"], kw["dt"], vote)
    assert orc.run_stages(1, 5) == 0
    assert sim.counters().interactions == orc.scalars()["interactions"]
    g, o = sim.accel(), orc.accel()
    if n > 1:
        assert rel_err(g, o).max() <= 1e-5
    else:
        assert np.all(g == 0)
    assert np.array_equal(sim.probe_accel(), sim.probe_accel())
    sim.close()
