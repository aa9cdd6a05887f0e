"""State in and vertices out with the largest pieces (1 MiB from 524,288 bodies:
32,768 bodies of position and velocity, 37,440 of state) and with all eight
workers (from 917,504 bodies), and rows for the network on both sides of the size
from which the runtime copies them. Copies are exact."""
import numpy as np
import pytest

from helpers import make_sim, random_model
from test_gpu_transfers import KW, _check, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [524_287, 524_288, 524_289, 917_504, 1_100_003])
def test_round_trip(nb, n):
    a, b = _state(n, n), _state(n, n + 1)
    sim = make_sim(a, **KW)
    _check(sim, a)
    sim.set_state(*b)
    _check(sim, b)
    sim.close()


@pytest.mark.parametrize("n", [2048, 70_001])
@pytest.mark.parametrize("rows", [5461, 5462, 30_000])
def test_rows_in_one_call_and_in_pieces(nb, rows, n):
    """Rows go in through slots below 512 KiB (5,461 rows of 24 floats) and by the
    runtime's copy from there: one call gives what small calls give."""
    from nbody_amd import universe as U

    sim = make_sim(U.uniform_ball(n, seed=2), vote_width=64, **KW)
    sim.set_model(random_model(6))
    x = np.random.default_rng(rows).normal(size=(rows, 24)).astype(np.float32)
    pieces = [sim.mlp_forward(x[i:i + 500]) for i in range(0, rows, 500)]
    assert np.array_equal(sim.mlp_forward(x), np.concatenate(pieces))
    sim.close()
