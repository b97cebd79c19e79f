"""The interp kernel at the edges of its launch rules, against the oracle.

A sample sums up to kw^d products of random sign, rounded four times each, in
32 bits on both sides: rel-L2 <= 2 * (4 + sqrt(kw^d / 2)) * 2^-24, at most
2.0e-6 for the 343 taps of kernel width 7 in 3-D.
"""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu

# name, image, osf, kernel width, sector width, samples, coils, lookup
CASES = [
    ("2d_one_sample", (16, 16), 1.0, 3, 8, 1, 1, 0),
    # coil groups of 1, 2, 4 and 8 and one coil past them; part of a wave's
    # samples; several chunks of a sector
    ("2d_2_coils", (17, 33), 1.0, 3, 8, 2000, 2, 0),
    ("2d_3_coils_kw1", (24, 40), 1.0, 1, 8, 65, 3, 0),
    ("2d_9_coils_kw2", (24, 40), 1.25, 2, 8, 900, 9, 1),
    ("2d_6_coils_kw5", (40, 52), 1.25, 5, 5, 9000, 6, 1),
    # padded sector longer than the grid; wider than a wave's row
    ("2d_short_grid_kw7", (9, 8), 1.0, 7, 4, 700, 8, 1),
    ("2d_wide_sector", (100, 90), 1.0, 4, 70, 3000, 1, 0),
    ("2d_sector_of_one", (20, 16), 1.0, 3, 1, 500, 4, 0),
    ("3d_chunks", (17, 9, 5), 1.0, 3, 8, 9000, 5, 0),
    ("3d_short_grid_kw6", (5, 4, 3), 1.5, 6, 4, 500, 8, 1),
    # one coil of the padded sector is what fits
    ("3d_wide_sector", (26, 25, 24), 1.0, 3, 23, 700, 3, 0),
    ("3d_kw7", (20, 18, 11), 1.5, 7, 8, 600, 2, 1),
    ("3d_kw4_odd_sector", (14, 16, 18), 1.5, 4, 5, 900, 16, 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_interp_edges(oracle, case):
    import torch
    name, img, osf, kw, sw, M, C, lookup = case
    print("case", name, flush=True)
    d = len(img)
    rng = np.random.default_rng(M + C)
    traj = rng.uniform(-0.5, 0.5, (d, M))
    traj[:, : M // 4] = np.round(traj[:, : M // 4] * 32) / 32  # grid points, sector edges, -1/2
    traj = np.clip(traj, -0.5, 0.4999).astype(np.float32)
    pl = capi.Plan(img, kw, sw, osf, lookup)
    pl.set_trajectory(torch.from_numpy(traj).cuda())
    ref = oracle.precompute(traj, img, osf, kw, sw, lookup=lookup, order="stable")
    gi = ref["info"]
    grid = W.complex_normal(rng, (C,) + oracle.grid_shape(gi))
    want = oracle.interp(gi, lookup, oracle.load_lut(osf, kw, lookup), ref["traj_sorted"], grid,
                         ref["sector_data_count"], ref["sector_centers"])
    tol = 2 * (4 + np.sqrt(kw ** d / 2)) * 2.0 ** -24
    for per_cu in (0, 1, 8):
        pl.set_workgroups_per_cu(per_cu)
        out = torch.full((C, M), float("nan"), dtype=torch.complex64, device="cuda")
        pl.interp_sorted(torch.from_numpy(grid).cuda(), out, C)
        assert oracle.rel_l2(out.cpu().numpy(), want) < tol, per_cu
