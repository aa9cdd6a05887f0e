"""The force traversal on both sides of every number of bodies at which the
number of waves per group changes (36,864, 114,688 and 409,600 bodies at width 64,
40,960 at the narrow widths: 576, 1,792, 6,400 and 640 groups of 64), with a last group that is full, holds one body, or ends
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
@pytest.mark.parametrize("n", [1, 63, 36_864, 36_865, 40_960, 40_961, 114_688, 114_715, 409_600, 409_601])
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


def _nests():
    """Every cell of level 3 nests: seven of its octants hold a pair of bodies, the
    last one the next level, down to level 18. 512 nests of 224 bodies, and 8
    bodies that pin the root."""
    signs = np.array([[1 if o >> k & 1 else -1 for k in range(3)] for o in range(8)], float)
    c = np.zeros((1, 3))
    h = 1.0
    for _ in range(3):
        h /= 2
        c = (c[:, None] + h * signs).reshape(-1, 3)
    out = [signs]
    for _ in range(16):
        mid = (c[:, None] + h / 2 * signs[:7]).reshape(-1, 3)
        out += [mid - h / 8, mid + h / 8]
        c, h = c + h / 2, h / 2
    return np.concatenate(out).astype(np.float32)


def test_walk_that_opens_deep_cells_everywhere(nb):
    """At an opening angle near 0 a wave pushes seven cells more than it takes in
    each of its first visits, so four waves (1,793 groups) have more left than they
    deal out again. Every body meets every body: the direct sum, within the FP32
    rounding of the terms (1e-5, as above)."""
    x = _nests()
    n = len(x)
    m = np.full(n, 1.0 / n, np.float32)
    v = np.zeros(n, np.float32)
    st = (x[:, 0].copy(), x[:, 1].copy(), x[:, 2].copy(), v, v.copy(), v.copy(), m)
    sim = make_sim(st, vote_width=64, theta=1e-7, softening=0.05, dt=1e-3)
    for s in range(1, 6):
        sim.run_stage(s)
    assert sim.counters().interactions == n * n
    idx = np.arange(0, n, 97, dtype=np.int32)
    assert rel_err(sim.accel()[idx], sim.direct_accel(idx)).max() <= 1e-5
    sim.close()
