"""The exact potential, which works out every pair once, at the edges of its
blocks (64 targets), tiles (256 sources), source chunks (n / 64) and target
batches (65,536), against FP64 sums over all ordered pairs by torch.

Bar: 1e-12 relative, the bar of the direct sum's accelerations (the terms'
relative error is below 1e-13 and all have one sign).
"""
import numpy as np
import pytest
import torch

from helpers import make_sim

pytestmark = pytest.mark.gpu


def _potential(st, soft):
    p = torch.from_numpy(np.stack(st[:3], 1).astype(np.float64)).cuda()
    m = torch.from_numpy(np.asarray(st[6], np.float64)).cuda()
    eps2 = float(np.float32(soft) * np.float32(soft))
    pe = 0.0
    for i in range(0, len(m), 512):
        r2 = torch.full((min(512, len(m) - i), len(m)), eps2, dtype=torch.float64, device="cuda")
        for k in range(3):
            r2 += (p[i:i + 512, k][:, None] - p[None, :, k]) ** 2
        inv = r2.rsqrt_()
        rows = torch.arange(inv.shape[0], device="cuda")
        inv[rows, i + rows] = 0.0
        pe -= 0.5 * float((inv * m[None, :] * m[i:i + 512, None]).sum())
    return pe


@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 257, 4096, 4097, 16_449, 65_536, 65_537, 65_700])
def test_exact_potential_at_edges(nb, n):
    from nbody_amd import universe as U

    st = U.halo_disk(n, seed=n % 83)
    sim = make_sim(st, theta=0.5, softening=0.03, dt=1e-3, vote_width=64)
    ref = _potential(st, 0.03)
    got = sim.diagnostics(0)["potential"]
    assert abs(got - ref) <= 1e-12 * abs(ref), (got, ref)
    assert sim.diagnostics(0)["potential"] == got
    sim.close()
