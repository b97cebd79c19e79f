"""The sector-width autotuner times the operator's own coil count (the kernels'
coil groups follow it), alone and among copies of itself."""

import pytest

from gpunufft_amd import autotune, capi
from gpunufft_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims, kw, widths, fill, coils", [
    ((96, 96), 3, (4, 8, 16), 4096, 1),
    ((64, 96), 5, (8, 16), 4096, 6),
    ((301, 250), 3, (8, 16), 4096, 3),     # (rocFFT)
    ((96, 96), 3, (8, 100), 4096, 4),      # a width that a batch refuses
    ((24, 20, 28), 3, (4, 8), 4096, 2),
    ((96, 96), 3, (8, 16), 0, 6),
])
def test_operator_is_timed_with_its_own_coils(monkeypatch, dims, kw, widths, fill, coils):
    import torch
    seen = []

    def note(cls, name, get):
        real = getattr(cls, name)
        monkeypatch.setattr(cls, name, lambda self, *a, **k: (seen.extend(get(a)), real(self, *a, **k))[1])

    note(capi.Batch, "__init__", lambda a: a[1])
    note(capi.Plan, "interp_sorted", lambda a: [a[2]])
    note(capi.Plan, "spread_sorted", lambda a: [a[2]])
    monkeypatch.setattr(autotune, "_CACHE", {})
    t = W.spiral_2d(8, 512, n_turns=8) if len(dims) == 2 else W.koosh_3d(64, 48)
    traj, dens = torch.from_numpy(t).cuda(), torch.from_numpy(W.ramp_density(t)).cuda()
    assert autotune.best_sector_width(dims, kw, 1.5, traj, dens, coils, widths=widths, fill_blocks=fill) in widths
    assert seen and set(seen) == {coils}
