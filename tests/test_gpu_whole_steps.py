"""Steps taken in one call (the force pass advances the bodies) against the same
steps with a launch per stage (timing on): bit for bit the same state,
accelerations and order."""
import numpy as np
import pytest

from helpers import make_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("n,vote", [(1, 16), (65, 64), (4097, 16), (50_001, 32), (120_003, 64)])
def test_whole_steps_equal_stages(nb, n, vote, fp64):
    from nbody_amd import _lib, universe as U

    st = U.rotating_disk(n, seed=n % 31) if n > 1 else tuple(np.full(1, v, np.float32) for v in (.1, .2, .3, 1, 2, 3, 1))
    kw = dict(theta=0.8, softening=0.05, dt=5e-3, vote_width=vote, flags=_lib.NB_FP64_POSITIONS if fp64 else 0)
    a, b = make_sim(st, **kw), make_sim(st, **kw)
    b.set_timing(True)
    for _ in range(2):
        a.steps(2)
        b.steps(2)
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
        assert np.array_equal(a.accel(), b.accel())
        assert np.array_equal(a.sorted(), b.sorted())
    a.close()
    b.close()
