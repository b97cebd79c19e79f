"""GNUFFT_LANE_PER_CU is the default of gnufft_plan_set_workgroups_per_cu.

The target is not in the results, except for the last bits of a CG solve on an odd
grid (it sizes the coil blocks, whose float sums set the fixed-point step): with a
wide sector a target of 8 gives other bits than the built-in one, and the
variable has to give the bits of the call.
"""

import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SOLVE = """
import sys
import numpy as np, torch
from gpunufft_amd import capi, workloads as W
dims, C = (30, 50), 4
rng = np.random.default_rng(2)
dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
traj = W.radial_2d(50, 100, golden=True)
p = capi.Plan(dims, 3, 32, 1.5)  # a grid of 45 x 75 points
if int(sys.argv[1]):
    p.set_workgroups_per_cu(int(sys.argv[1]))
p.set_trajectory(dev(traj), dev(W.ramp_density(traj)))
p.set_sens(dev(W.gaussian_sens(dims, C, seed=1)), C)
x = torch.empty((1, 50, 30), dtype=torch.complex64, device="cuda")
capi.CGSense(p, C, 1e-3).solve(dev(W.complex_normal(rng, (C, traj.shape[1]))), x, 8)
torch.cuda.synchronize()
sys.stdout.write(x.cpu().numpy().tobytes().hex())
"""


def _solve(target, env):
    e = {k: v for k, v in os.environ.items() if k != "GNUFFT_LANE_PER_CU"}
    e.update(env)
    r = subprocess.run([sys.executable, "-c", SOLVE, str(target)], env=e, capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.strip()


def test_environment_sets_the_default():
    plain, call = _solve(0, {}), _solve(8, {})
    assert len(plain) == len(call) == 50 * 30 * 16
    assert plain != call
    assert _solve(0, {"GNUFFT_LANE_PER_CU": "8"}) == call
    assert _solve(8, {"GNUFFT_LANE_PER_CU": "1"}) == call  # the plan's own target goes first
    assert _solve(0, {"GNUFFT_LANE_PER_CU": "99"}) == plain  # out of range: ignored
