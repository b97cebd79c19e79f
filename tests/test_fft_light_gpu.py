"""FFT passes of small grids (few tiles) and of short lines at the edges of their
tiles: the light and the short-line kernels run the same stages in the same
order as the full tiles that a batch uses, so a plan by itself and a batch of
that plan give the same bits (for lengths without kernels of their own, which a
batch does not use).
"""

import numpy as np
import pytest

from gpunufft_amd import capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu

# image, osf, coils, sensitivities: 128 .. 1024 threads per tile, partial tiles
# in x, one image line, prime stages, 3-D with few tiles
CASES = [
    ((16, 16), 1.0, 1, False),
    ((64, 64), 2.0, 1, True),
    ((65, 66), 2.0, 3, True),
    ((250, 9), 1.5, 2, False),
    ((9, 250), 1.5, 2, True),
    ((240, 240), 2.0, 12, True),
    ((256, 100), 2.0, 16, True),
    ((500, 500), 2.0, 2, False),
    ((143, 152), 1.0, 5, True),
    ((480, 450), 2.0, 9, True),
    ((24, 20, 18), 1.5, 2, True),
    # short lines with many tiles: 66 points in y, 22 and 4 in z
    ((100, 44, 176), 1.5, 3, True),
    ((165, 110, 22), 1.0, 8, False),
    ((165, 100, 4), 1.0, 12, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + "_c%d" % c[2])
def test_small_grids_match_batch(case):
    import torch
    img, osf, C, with_sens = case
    print("case", case, flush=True)
    rng = np.random.default_rng(sum(img) + C)
    d, M = len(img), 3000
    traj = rng.uniform(-0.5, 0.5, (d, M)).astype(np.float32)
    pl = capi.Plan(img, 3, 8, osf)
    pl.set_trajectory(torch.from_numpy(traj).cuda())
    shape = tuple(reversed(img))
    if with_sens:
        sens = torch.from_numpy(W.complex_normal(rng, (C,) + shape)).cuda()
        pl.set_sens(sens, C)
    n_img = 1 if with_sens else C
    k = torch.from_numpy(W.complex_normal(rng, (C, M))).cuda()
    x = torch.from_numpy(W.complex_normal(rng, (n_img,) + shape)).cuda()
    pl.set_fft(0)
    out = [torch.full((n_img,) + shape, float("nan"), dtype=torch.complex64, device="cuda") for _ in range(2)]
    fwd = [torch.full((C, M), float("nan"), dtype=torch.complex64, device="cuda") for _ in range(2)]
    pl.adjoint(k, out[0], C)
    pl.forward(x, fwd[0], C)
    b = capi.Batch([pl], [C])
    b.adjoint([k], [out[1]])
    b.forward([x], [fwd[1]])
    torch.cuda.synchronize()
    assert torch.isfinite(torch.view_as_real(out[0])).all()
    assert torch.equal(torch.view_as_real(out[0]), torch.view_as_real(out[1]))
    assert torch.equal(torch.view_as_real(fwd[0]), torch.view_as_real(fwd[1]))
