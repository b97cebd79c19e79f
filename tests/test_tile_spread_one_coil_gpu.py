"""The tile spread of one coil (sub-tiles of eight points in x, rounds of 64
samples) at the edges of its tiles, against the oracle, with the bound of the other
coil counts; and a batch of one-coil plans against the plans by themselves."""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W
from test_tile_spread_gpu import TOL, _traj

pytestmark = pytest.mark.gpu

# name, image, osf, kernel width, sector width, samples, lookup, trajectory
CASES = [
    ("2d_round", (17, 33), 1.0, 3, 8, 64, 0, "uniform"),
    ("2d_round_plus_1", (24, 40), 1.0, 3, 8, 65, 0, "uniform"),
    ("2d_short_grid_kw7", (9, 8), 1.0, 7, 4, 700, 1, "uniform"),
    ("2d_chunks", (48, 31), 2.0, 3, 8, 30000, 0, "centre"),
    ("2d_kw5", (40, 52), 1.25, 5, 5, 9000, 1, "centre"),
    ("3d_tile_plus_1", (17, 9, 5), 1.0, 3, 8, 129, 0, "uniform"),
    ("3d_short_grid_kw4", (5, 4, 3), 1.5, 4, 4, 500, 1, "uniform"),
    ("3d_kw6_chunks", (20, 18, 11), 1.5, 6, 4, 9000, 1, "centre"),
    ("3d_kw1", (24, 20, 17), 1.0, 1, 8, 900, 0, "uniform"),
    ("3d_dense", (16, 16, 16), 1.5, 3, 8, 60000, 0, "uniform"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_one_coil(oracle, case):
    import torch
    name, img, osf, kw, sw, M, lookup, kind = case
    print("case", name, flush=True)
    rng = np.random.default_rng(M)
    traj = _traj(rng, len(img), M, kind)
    pl = capi.Plan(img, kw, sw, osf, lookup)
    pl.set_trajectory(torch.from_numpy(traj).cuda())
    ref = oracle.precompute(traj, img, osf, kw, sw, lookup=lookup, order="stable")
    data = W.complex_normal(rng, (1, M))
    want = oracle.spread(ref["info"], lookup, oracle.load_lut(osf, kw, lookup), ref["traj_sorted"], data,
                         ref["sector_data_count"], ref["sector_centers"])
    grid = torch.full((1,) + want.shape[1:], float("nan"), dtype=torch.complex64, device="cuda")
    pl.spread_sorted(torch.from_numpy(data).cuda(), grid, 1)
    assert oracle.rel_l2(grid.cpu().numpy(), want) < TOL
    # the caller's order, and a batch (the same sums)
    k = torch.empty((1, M), dtype=torch.complex64, device="cuda")
    k[:, torch.from_numpy(ref["data_indices"].astype(np.int64)).cuda()] = torch.from_numpy(data).cuda()
    again = torch.full_like(grid, float("nan"))
    pl.adjoint(k, again, 1, capi.CONVOLUTION)
    assert torch.equal(torch.view_as_real(again), torch.view_as_real(grid))
    if kw == 1:  # (its deapodization is not finite)
        return
    shape = (1,) + tuple(reversed(img))
    alone, batched = (torch.full(shape, float("nan"), dtype=torch.complex64, device="cuda") for _ in range(2))
    pl.adjoint(k, alone, 1)
    capi.Batch([pl], [1]).adjoint([k], [batched])
    torch.cuda.synchronize()
    assert oracle.rel_l2(batched.cpu().numpy(), alone.cpu().numpy()) < 1e-6
