"""The tile spread and both ways of building its lists, against the oracle.

Tables are compared exactly. The spread's grid: a point sums n products of
random sign, each rounded four times; the partial sums' roundings add up to
about eps * sqrt(n / 2) of the result (eps = 2^-24; n <= 2000 here: 32 eps), in
the oracle (32-bit as well) and in the kernel: rel-L2 <= 2 * (32 + 4) eps =
4.3e-6.
"""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 72 * 2.0 ** -24


def _traj(rng, dim, M, kind):
    if kind == "centre":  # several chunks in the tiles around the centre
        t = rng.normal(0, 0.06, (dim, M))
    else:
        t = rng.uniform(-0.5, 0.5, (dim, M))
        t[:, : M // 4] = np.round(t[:, : M // 4] * 32) / 32  # grid points, tile edges, -1/2
    return np.clip(t, -0.5, 0.4999).astype(np.float32)


# name, image, osf, kernel width, sector width, samples, coils, lookup, trajectory
CASES = [
    # one sample; a block and one more of the short tables; grids of one tile,
    # of a tile and one point, shorter than a tile and the taps together
    ("2d_one_sample", (16, 16), 1.0, 3, 8, 1, 1, 0, "uniform"),
    ("2d_tile_plus_1", (17, 33), 1.0, 3, 8, 129, 2, 0, "uniform"),
    ("2d_short_grid_kw7", (9, 8), 1.0, 7, 4, 700, 9, 1, "uniform"),
    ("2d_kw1", (24, 40), 1.0, 1, 8, 900, 4, 0, "uniform"),
    ("2d_chunks", (48, 31), 2.0, 3, 8, 30000, 5, 0, "centre"),
    ("2d_kw5_chunks", (40, 52), 1.25, 5, 5, 9000, 8, 1, "centre"),
    ("3d_tile_plus_1", (17, 9, 5), 1.0, 3, 8, 128, 3, 0, "uniform"),
    ("3d_short_grid_kw4", (5, 4, 3), 1.5, 4, 4, 500, 8, 1, "uniform"),
    ("3d_kw6_chunks", (20, 18, 11), 1.5, 6, 8, 9000, 2, 1, "centre"),
    # more keys than the short tables take: sorted by the library
    ("3d_long_tables", (80, 80, 40), 1.5, 3, 4, 20000, 1, 0, "centre"),
    ("2d_long_tables", (600, 500), 1.0, 3, 4, 20001, 3, 0, "centre"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tables_and_spread(oracle, case):
    import torch
    name, img, osf, kw, sw, M, C, lookup, kind = case
    print("case", name, flush=True)
    rng = np.random.default_rng(M + C)
    traj = _traj(rng, len(img), M, kind)
    dens = rng.uniform(0.1, 1, M).astype(np.float32)
    pl = capi.Plan(img, kw, sw, osf, lookup)
    pl.set_trajectory(torch.from_numpy(traj).cuda(), torch.from_numpy(dens).cuda())
    t = pl.tables()
    ref = oracle.precompute(traj, img, osf, kw, sw, dens, lookup=lookup)
    assert np.array_equal(pl.assigned_sectors(), ref["sectors"])
    for k in ("sector_data_count", "sector_centers", "data_indices", "traj_sorted", "dens_sorted"):
        assert np.array_equal(t[k], ref[k]), k
    # spread of samples in (stable) sector order
    ref = oracle.precompute(traj, img, osf, kw, sw, lookup=lookup, order="stable")
    data = W.complex_normal(rng, (C, M))
    want = oracle.spread(ref["info"], lookup, oracle.load_lut(osf, kw, lookup), ref["traj_sorted"], data,
                         ref["sector_data_count"], ref["sector_centers"])
    grid = torch.full((C,) + want.shape[1:], float("nan"), dtype=torch.complex64, device="cuda")
    pl.spread_sorted(torch.from_numpy(data).cuda(), grid, C)
    assert oracle.rel_l2(grid.cpu().numpy(), want) < TOL
