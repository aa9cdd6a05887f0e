"""State in and vertices out with the largest pieces (1 MiB from 524,288 bodies:
32,768 bodies of position and velocity, 37,440 of state) and with all eight
workers (from 917,504 bodies). Copies are exact."""
import pytest

from helpers import make_sim
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
