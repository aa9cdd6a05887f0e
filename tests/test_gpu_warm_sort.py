"""The sort of a warm build (bodies bucketed by the last tree's keys, each
bucket sorted by one block) at its edges: fewer bodies than a bucket, whole
buckets and one more, a bucket at the limit of the LDS sort and past it, and
runs of bodies that share their first 21 octants inside a bucket, up to runs
that fill one and runs that make it too large for LDS.

Every body's path and depth and the sorted order are integers: they equal the
oracle's.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim

pytestmark = pytest.mark.gpu


def _moving(n, run, seed):
    """n bodies in [-1, 1]^3 (masses 1e-9: gravity moves none by a rounding)
    drifting at up to 1, of which `run` rest within 2e-7 of one point: a cell
    of level 21 is 9.5e-7 wide, and the FP32 spacing there is 9e-10."""
    g = np.random.default_rng(seed)
    p = g.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    v = g.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    at = g.permutation(n)[:run]
    base = np.array([0.0123, -0.0117, 0.0109])
    close = (base + g.uniform(0.0, 2e-7, (4 * run + 1, 3))).astype(np.float32)
    p[at] = np.unique(close, axis=0)[g.permutation(run)]
    v[at] = 0.0
    return p, v, np.full(n, 1e-9, np.float32)


@pytest.mark.parametrize("n,run", [(1, 0), (2, 0), (2, 2), (255, 0), (256, 0), (257, 2), (512, 16), (513, 17),
                                   (700, 300), (1025, 512), (1500, 700), (9001, 64)])
def test_warm_sort_edges(nb, oracle, n, run):
    p, v, m = _moving(n, run, seed=n + run)
    st = tuple(np.ascontiguousarray(a) for a in (*p.T, *v.T, m))
    sim = make_sim(st, theta=0.5, softening=0.05, dt=0.02)
    for _ in range(2):
        sim.steps(1)
        x, y, z, vx, vy, vz = sim.state()
        orc = make_oracle((x, y, z, vx, vy, vz, m), 0.5, 0.05, 0.02, 16)
        for stage in range(1, 5):
            sim.run_stage(stage)
        assert orc.run_stages(1, 2) == 0
        gp, gd = sim.paths()
        op, od = orc.paths()
        assert np.array_equal(gd, od) and gd.min() > 0
        assert np.array_equal(gp, op)
        assert orc.run_stages(3, 4) == 0
        assert np.array_equal(sim.sorted(), orc.sorted())
    sim.close()
