"""The coarse traversal on both sides of every number of bodies at which the
number of waves per group changes (20,480, 81,920 and 589,824 bodies: 320, 1,280
and 9,216 groups of 64), and its listed-group passes through training.

The oracle takes the same opening decisions: equal interaction counts (through
the features' exact counts and the counter), accelerations within 1e-5, as in
the tests of the other sizes. The bodies have moved for two steps, so the
relative test takes part.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim, rel_err

pytestmark = pytest.mark.gpu

THETA_C, ALPHA, EPS = 0.9, 0.03, 0.02


@pytest.mark.parametrize("n", [64, 65, 20_480, 20_481, 81_920, 81_921, 98_331, 327_699, 589_824, 589_849])
def test_coarse_at_split_edges(nb, oracle, n):
    from nbody_amd import universe as U

    st = U.plummer(n, seed=n % 89)
    sim = make_sim(st, theta=0.4, softening=EPS, dt=1e-3, vote_width=64, coarse_theta=THETA_C, coarse_alpha=ALPHA,
                   method=nb._lib.NB_MODE_COARSE)
    sim.steps(2)
    x, y, z, vx, vy, vz = sim.state()
    orc = make_oracle((x, y, z, vx, vy, vz, st[6]), 0.4, EPS, 1e-3, 64, flags=1)
    a = sim.accel()
    orc.set_accel(*(np.ascontiguousarray(a[:, j]) for j in range(3)), sim.counters().step)
    for s in range(1, 6):
        sim.run_stage(s)
    assert orc.run_stages(1, 4) == 0
    orc.moments()
    srt = orc.sorted()
    assert np.array_equal(srt, sim.sorted())
    oa, _, _, ni = orc.coarse(THETA_C, features=False, alpha=ALPHA)
    assert sim.counters().interactions == ni
    assert rel_err(sim.accel()[srt], oa[:n]).max() <= 1e-5
    assert np.array_equal(sim.probe_accel(), sim.probe_accel())
    sim.close()


@pytest.mark.parametrize("groups", [1, 320, 321, 1536, 1537])
def test_training_on_listed_groups(nb, groups):
    """Two trainings on the same bodies give the same network bit for bit,
    whatever number of waves works on the sampled groups."""
    from nbody_amd import universe as U

    st = U.gaussian_clusters(131_072, seed=4)
    blobs = []
    for _ in range(2):
        sim = make_sim(st, theta=0.4, softening=EPS, dt=1e-3, vote_width=64, coarse_theta=THETA_C,
                       coarse_alpha=ALPHA, method=nb._lib.NB_MODE_LEARNED)
        rep = sim.train(steps=2, groups_per_step=groups, iters=20, batch=256, seed=3)
        assert rep["samples"] == 2 * groups * 64 and np.isfinite(rep["loss_last"])
        blobs.append(sim.get_model())
        sim.close()
    assert np.array_equal(blobs[0], blobs[1])
