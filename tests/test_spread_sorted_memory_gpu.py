"""gnufft_spread_sorted needs no device memory beyond what the adjoint of as many
coils needs: after one, it allocates nothing (a trajectory that is long for its
grid would take the most), and it can be captured into a graph."""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu


def _plan(M, C):
    import torch
    rng = np.random.default_rng(M)
    p = capi.Plan((32, 32), 3, 8, 2.0)
    p.set_trajectory(torch.from_numpy(rng.uniform(-0.5, 0.4999, (2, M)).astype(np.float32)).cuda())
    data = torch.from_numpy(W.complex_normal(rng, (C, M))).cuda()
    p.adjoint(data, torch.empty((C, 32, 32), dtype=torch.complex64, device="cuda"), C)
    torch.cuda.synchronize()
    return torch, p, data, torch.empty((C, 64, 64), dtype=torch.complex64, device="cuda")


@pytest.mark.parametrize("M", [200000, 1 << 20], ids=["short_tables", "long_tables"])
def test_no_memory_beyond_the_adjoint(M):
    torch, p, data, grid = _plan(M, 8)
    before = torch.cuda.mem_get_info()[0]
    p.spread_sorted(data, grid, 8)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 1 << 20


def test_captured_after_an_adjoint():
    torch, p, data, grid = _plan(30000, 3)
    want = torch.empty_like(grid)
    p.spread_sorted(data, want, 3)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        p.spread_sorted(data, grid, 3)
    for rep in range(3):
        grid.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(grid), torch.view_as_real(want)), rep
        p.adjoint(data, torch.empty((3, 32, 32), dtype=torch.complex64, device="cuda"), 3)
