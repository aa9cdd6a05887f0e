"""Builds that stop with an error: a pool too small for the tree, found by the
kernel that links the cells, and bodies that only separate between levels 65 and
83, found by the binary tree (those on one 84-level path are found before, by the
sort). In a first build and in a warm one; below 524,288 bodies, where the
build's own blocks scan and group the cells, and above; with splitters by
sampling, and by radix passes.

The step reports the status, the steps queued behind it change nothing, and the
handle goes on with its next state: paths and order equal the oracle's.
"""
import numpy as np
import pytest

from helpers import make_oracle, make_sim

pytestmark = pytest.mark.gpu

KW = dict(theta=0.8, softening=0.05, dt=1.0, pool_factor=1.0)
SIZES = [20_000, 100_002, 200_002, 600_002]


def _state(p, v):
    """Bodies without mass: nothing accelerates, positions after a step are x + v dt."""
    return tuple(np.ascontiguousarray(a, np.float32) for a in (*p.T, *v.T, np.zeros(len(p))))


def _pool(n, warm):
    """Pairs a few 1e-6 apart in a box of 2: a chain of about a dozen cells each.
    Warm: each pair's second body comes there in one step."""
    g = np.random.default_rng(n)
    p, v = np.empty((n, 3)), np.zeros((n, 3))
    p[0::2] = g.uniform(-1.0, 1.0, (n // 2, 3))
    p[1::2] = p[0::2] + g.uniform(2e-6, 4e-6, (n // 2, 3))
    if warm:
        far = g.uniform(-1.0, 1.0, (n // 2, 3))
        v[1::2] = p[1::2] - far
        p[1::2] = far
    return _state(p, v)


def _deep(n, warm):
    """A box around 0 of half size 1 and, in each octant at 0, two bodies that
    separate at level 71. Warm: the second comes there from level 56; every
    sum is exact in FP32."""
    g = np.random.default_rng(n)
    p, v = g.uniform(-1.0, 1.0, (n, 3)), np.zeros((n, 3))
    corners = np.stack(np.meshgrid([-1.0, 1.0], [-1.0, 1.0], [-1.0, 1.0]), -1).reshape(8, 3)
    at = g.permutation(n)[:24].reshape(3, 8)
    p[at[0]] = corners
    p[at[1]] = corners * 1.25 * 2.0 ** -70
    p[at[2]] = corners * 1.75 * 2.0 ** -70
    if warm:
        v[at[2]] = p[at[2]] - corners * 2.0 ** -55
        p[at[2]] = corners * 2.0 ** -55
    return _state(p, v)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("kind", ["pool", "deep"])
def test_build_error_and_recovery(nb, oracle, kind, warm, n):
    bad = _pool(n, warm) if kind == "pool" else _deep(n, warm)
    sim = make_sim(bad, **KW)
    if warm:
        sim.steps(1)
    before = sim.state()
    with pytest.raises(nb.NbError) as e:
        sim.steps(3)
    assert e.value.code == (nb._lib.NB_E_POOL if kind == "pool" else nb._lib.NB_E_DEPTH)
    for a, b in zip(sim.state(), before):
        assert np.array_equal(a, b)
    g = np.random.default_rng(n + 1)
    good = _state(g.uniform(-1.0, 1.0, (n, 3)), g.uniform(-1e-3, 1e-3, (n, 3)))
    sim.set_state(*good)
    sim.steps(1)
    x, y, z, vx, vy, vz = sim.state()
    orc = make_oracle((x, y, z, vx, vy, vz, good[6]), 0.8, 0.05, 1.0, 16)
    for stage in range(1, 5):
        sim.run_stage(stage)
    assert orc.run_stages(1, 2) == 0
    gp, gd = sim.paths()
    op, od = orc.paths()
    assert np.array_equal(gd, od) and np.array_equal(gp, op)
    assert orc.run_stages(3, 4) == 0
    assert np.array_equal(sim.sorted(), orc.sorted())
    sim.close()
