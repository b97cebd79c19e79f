"""CG-SENSE on grids with an odd length.

There the forward's and the adjoint's shifts differ, the two are not adjoint to
each other, and CG amplifies rounding: what a solve returns is settled by the
order and the precision of the adjoint's sums. The expected images
(golden/cg_odd_grids.npz) come from this library's gridding by padded sectors,
fixed-point sums and a fold; a solver on any other sums ends up 4e-3 to 8e-2
from them here. The bound is that of a result in 32 bits, 2e-5.
"""

import os

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 2e-5

# name: image, osf, kernel width, coils, lookup, seeds of inputs and of coil maps
CASES = {
    "2d_kw3": ((50, 34), 1.5, 3, 3, 1, 101, 1),
    "2d_kw4": ((29, 40), 1.5, 4, 6, 0, 402, 2),
    "3d_kw3": ((18, 14, 10), 1.5, 3, 3, 0, 700, 0),
    "3d_kw5": ((14, 13, 15), 1.5, 5, 2, 1, 801, 1),
}


@pytest.mark.parametrize("name", CASES)
def test_cg_on_odd_grid(oracle, name):
    import torch
    dims, osf, kw, C, lookup, seed, sens_seed = CASES[name]
    print("case", name, flush=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    rng = np.random.default_rng(seed)
    n = max(dims)
    traj = W.radial_2d(n, 2 * n, golden=True) if len(dims) == 2 else W.koosh_3d(n * n // 2, 2 * n)
    dens = W.ramp_density(traj, len(dims) - 1)
    kd = dev(W.complex_normal(rng, (C, traj.shape[1])))
    p = capi.Plan(dims, kw, 8, osf, lookup)
    p.set_sens(dev(W.gaussian_sens(dims, C, seed=sens_seed)), C)
    p.set_trajectory(dev(traj), dev(dens))
    assert any(g % 2 for g in p.info().grid[:len(dims)])
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "cg_odd_grids.npz"), allow_pickle=False) as f:
        want = f[name]
    cg = capi.CGSense(p, C, 1e-3)
    x = torch.empty(want.shape, dtype=torch.complex64, device="cuda")
    for use_graph in (False, True, True):
        x.zero_()
        cg.solve(kd, x, 10, use_graph)
        torch.cuda.synchronize()
        assert oracle.rel_l2(x.cpu().numpy(), want) < TOL, use_graph
    # another trajectory of the plan, and the first one again
    p.set_trajectory(dev(np.ascontiguousarray(-traj[:, ::-1]).clip(-0.5, 0.4999)), dev(dens))
    cg.solve(kd, x, 2)
    p.set_trajectory(dev(traj), dev(dens))
    cg.solve(kd, x, 10)
    torch.cuda.synchronize()
    assert oracle.rel_l2(x.cpu().numpy(), want) < TOL
