"""State in and out of the engine at the edges of the pieces it is moved in (256
KiB below 65,536 bodies, 512 KiB from there: 8,192 and 16,384 bodies of position
and velocity, 9,344 and 18,688 bodies of state), with several workers, with
either output left out, and from two threads at once on two handles. Copies are
exact."""
import threading

import numpy as np
import pytest

from helpers import make_sim, random_model

pytestmark = pytest.mark.gpu

KW = dict(theta=0.5, softening=0.05, dt=1e-3)


def _state(n, seed):
    g = np.random.default_rng(seed)
    return tuple(g.normal(size=n).astype(np.float32) for _ in range(6)) + (g.uniform(0.5, 1.0, n).astype(np.float32),)


def _check(sim, st):
    n = len(st[0])
    for got, put in zip(sim.state(), st):
        assert np.array_equal(got, put)
    one = np.ones(n, np.float32)
    pos, vel = np.full((n, 4), 7, np.float32), np.full((n, 4), 7, np.float32)
    want_p, want_v = np.stack([*st[:3], one], 1), np.stack([*st[3:6], one], 1)
    sim.copy_vertices(pos, vel)
    assert np.array_equal(pos, want_p) and np.array_equal(vel, want_v)
    pos[:], vel[:] = 7, 7
    sim.copy_vertices(pos, None)
    sim.copy_vertices(None, vel)
    assert np.array_equal(pos, want_p) and np.array_equal(vel, want_v)
    assert np.array_equal(sim.accel(), np.zeros((n, 3), np.float32))
    assert np.array_equal(sim.sorted(), np.arange(n))
    assert np.array_equal(sim.masses(), st[6])
    assert sim.counters().step == -1


@pytest.mark.parametrize("n", [1, 63, 8192, 8193, 9344, 9345, 32_768, 65_535, 65_536, 65_537, 149_505, 300_001])
def test_round_trip(nb, n):
    from nbody_amd import _lib

    a, b = _state(n, n), _state(n, n + 1)
    sim = make_sim(a, flags=_lib.NB_FP64_POSITIONS, **KW)
    _check(sim, a)
    sim.set_state(*b)
    sim.set_state(*a)  # twice: the pieces of the first may still be on their way
    _check(sim, a)
    assert np.array_equal(sim.positions64(), np.stack(a[:3], 1).astype(np.float64))
    sim.steps(1)
    sim.set_state(*b)
    _check(sim, b)
    sim.close()


def test_two_threads_two_handles(nb):
    states = [_state(200_003, 1), _state(150_001, 2)]
    sims = [make_sim(st, **KW) for st in states]
    bad = []

    def work(sim, st):
        try:
            for _ in range(5):
                sim.set_state(*st)
                _check(sim, st)
        except BaseException as e:  # reported by the main thread
            bad.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(sims, states)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    for s in sims:
        s.close()


def test_kept_scratch_is_not_seen(nb):
    """Gradients of several batch sizes in turn: the memory that one call leaves
    to the next holds nothing of it."""
    g = np.random.default_rng(5)
    st = _state(2048, 3)
    sims = [make_sim(st, vote_width=64, **KW) for _ in range(2)]
    model = random_model(4)
    for s in sims:
        s.set_model(model)
    for n in (64, 4096, 63, 20_000, 4096, 1):
        x, t = g.normal(size=(n, 24)).astype(np.float32), g.normal(size=(n, 3)).astype(np.float32)
        fresh = make_sim(st, vote_width=64, **KW)
        fresh.set_model(model)
        for s in sims:
            for got, want in zip(s.mlp_loss_grad(x, t), fresh.mlp_loss_grad(x, t)):
                assert np.array_equal(got, want)
            assert np.array_equal(s.mlp_adam(x, t, 3, 1e-3), fresh.mlp_adam(x, t, 3, 1e-3))
            assert np.array_equal(s.mlp_forward(x), fresh.mlp_forward(x))
        fresh.close()
    for s in sims:
        s.close()
