"""The FP32 training kernels at the edges of their tiles: one row, part of a
wave's 16 rows, one tile of 32 rows and its neighbours, as many tiles as blocks
run (256) and one more, so that a block takes a second tile.

Bars, as for the training kernels at other sizes: the loss within 1e-5 of the
FP64 oracle's, the gradient within 1e-4 of its largest component (sums of FP32
products over at most 16,449 rows, whose rounding stays near 1e-6 of it).
"""
import numpy as np
import pytest

from helpers import make_sim, random_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 32, 33, 64, 65, 128, 8192, 8193, 16_449])
def test_gradient_at_tile_edges(nb, oracle, rows):
    from nbody_amd import universe as U

    sim = make_sim(U.uniform_ball(256, seed=3), theta=0.4, softening=0.01, dt=1e-3, vote_width=64,
                   coarse_theta=0.9, method=nb._lib.NB_MODE_LEARNED)
    blob = random_model(rows)
    sim.set_model(blob)
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, 24)).astype(np.float32)
    t = rng.normal(size=(rows, 3)).astype(np.float32)
    loss, g = sim.mlp_loss_grad(x, t)
    oloss, og = oracle.mlp_loss_grad(blob[:5955].astype(np.float64), x, t)
    assert abs(loss - oloss) <= 1e-5 * abs(oloss)
    assert np.abs(g - og).max() <= 1e-4 * np.abs(og).max()
    again = sim.mlp_loss_grad(x, t)
    assert again[0] == loss and np.array_equal(again[1], g)
    sim.close()
