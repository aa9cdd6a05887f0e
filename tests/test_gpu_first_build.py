"""The first build of a state, which has no last order to start from: up to
131,072 bodies by buckets between sampled splitters (1024 samples up to 65,536
bodies, 2048 above), the radix sort beyond. Around those sizes and around whole
buckets of 128 bodies, on positions that fit the sampling (a ball, a lattice row
by row), that go against it (the bodies it reads in one corner, the others
elsewhere), and that make buckets too large for LDS (most bodies within a few
cells of level 21). Paths, depths and the order are integers and equal the
oracle's.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim

pytestmark = pytest.mark.gpu


def _positions(kind, n, g):
    if kind == "ball":
        return g.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    if kind == "unseen":
        # the bodies that a sample of 2048 reads near one corner: the others share a few buckets
        p = g.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
        i = np.arange(2048, dtype=np.uint64) * np.uint64(0x9E3779B1) & np.uint64(0xffffffff)
        at = np.unique((i * np.uint64(n) >> np.uint64(32)).astype(np.int64))
        p[at] = (np.array([0.9, 0.9, 0.9]) + 1e-3 * g.random((len(at), 3))).astype(np.float32)
        return p
    if kind == "lattice":
        k = round(n ** (1 / 3))
        x = np.linspace(-1.0, 1.0, k)
        return np.stack([a.ravel() for a in np.meshgrid(x, x, x, indexing="ij")], 1).astype(np.float32)
    # runs: 700 and more bodies sharing 21 levels, and copies of the rest nowhere
    p = g.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    k = min(n - 2, 900)
    close = np.unique((np.array([0.0123, -0.0117, 0.0109]) + g.uniform(0, 2e-7, (4 * k, 3))).astype(np.float32), axis=0)
    p[g.permutation(n)[:k]] = close[g.permutation(len(close))[:k]]
    return p


@pytest.mark.parametrize("kind,n", [("ball", n) for n in (1, 127, 128, 129, 1023, 65_536, 65_537, 131_071, 131_072, 131_073)]
                         + [("unseen", n) for n in (4096, 30_000, 65_536)] + [("lattice", n) for n in (1000, 32_768, 125_000)]
                         + [("runs", n) for n in (1000, 5000, 40_000)])
def test_first_build(nb, oracle, kind, n):
    g = np.random.default_rng(n)
    p = _positions(kind, n, g)
    zero, m = np.zeros(n, np.float32), np.full(n, 1.0 / n, np.float32)
    st = (*(np.ascontiguousarray(a) for a in p.T), zero, zero, zero, m)
    sim = make_sim(st, theta=0.8, softening=0.05, dt=1e-3)
    for _ in range(2):  # the second state on the same handle, in another order
        orc = make_oracle(st, 0.8, 0.05, 1e-3, 16)
        for stage in (1, 2):
            sim.run_stage(stage)
        assert orc.run_stages(1, 2) == 0
        gp, gd = sim.paths()
        op, od = orc.paths()
        assert np.array_equal(gd, od) and gd.min() > 0
        assert np.array_equal(gp, op)
        for stage in (3, 4):
            sim.run_stage(stage)
        assert orc.run_stages(3, 4) == 0
        assert np.array_equal(sim.sorted(), orc.sorted())
        assert sim.counters().large_buckets == 0  # counted for builds from a last order only
        order = g.permutation(n)
        st = tuple(np.ascontiguousarray(a[order]) for a in st)
        sim.set_state(*st)
    sim.close()
