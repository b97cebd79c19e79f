"""Short trajectory tables whose partial tiles exceed the plan's bound: longer chunks.

33 points along an axis are two tiles and a point. 2^18 samples whose seven taps
end past the last point meet three tiles per axis, nine in all: 2.36 M list
entries make 4608 chunks of 512, more than the 4096 partial tiles (a million points)
that the plan allows, and the chunks are doubled. A point sums up to 2^18 products
of random sign in 32 bits, in the oracle and in the kernel: rel-L2 <= 2 *
(sqrt(2^18 / 2) + 4) * 2^-24 = 4.4e-5.
"""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_chunks_are_doubled(oracle):
    import torch
    img, osf, kw, sw, M, C = (22, 22), 1.5, 7, 8, 1 << 18, 2
    rng = np.random.default_rng(8)
    traj = ((32 + rng.uniform(-0.4, 0.4, (2, M))) / 33 - 0.5).astype(np.float32)
    p = capi.Plan(img, kw, sw, osf)
    p.set_trajectory(torch.from_numpy(traj).cuda())
    ref = oracle.precompute(traj, img, osf, kw, sw, lookup=0, order="stable")
    data = W.complex_normal(rng, (C, M))
    want = oracle.spread(ref["info"], 0, oracle.load_lut(osf, kw, 0), ref["traj_sorted"], data,
                         ref["sector_data_count"], ref["sector_centers"])
    grid = torch.full((C,) + want.shape[1:], float("nan"), dtype=torch.complex64, device="cuda")
    p.spread_sorted(torch.from_numpy(data).cuda(), grid, C)
    assert oracle.rel_l2(grid.cpu().numpy(), want) < 2 * (np.sqrt(M / 2) + 4) * 2.0 ** -24
