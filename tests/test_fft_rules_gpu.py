"""Which kernels the passes of small transforms take: the light ones only where
they are not slower than the full tiles, which a batch always uses.

Both run the same stages in the same order, so on both sides of each line a plan
by itself and a batch of that plan give the same bits (lengths without kernels
of their own). At sizes where the light kernels take 1.3 to 1.5 times the full
tiles' time, a plan by itself takes no longer than a batch of it, which sends its
descriptors to the device besides (226 and 294 us at 608^2, 32 coils).
"""

import numpy as np
import pytest

from gpunufft_amd import capi

pytestmark = pytest.mark.gpu


def _setup(img, osf, C):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(sum(img) + C)
    rnd = lambda *s: torch.view_as_complex(torch.randn(s + (2,), generator=g, device="cuda"))
    shape = tuple(reversed(img))
    pl = capi.Plan(img, 3, 8, osf)
    pl.set_trajectory((torch.rand((len(img), 700), generator=g, device="cuda") - 0.5).contiguous())
    pl.set_sens(rnd(C, *shape), C)
    pl.set_fft(capi.FFT_FUSED)
    return torch, pl, rnd(C, 700), rnd(1, *shape)


# image, osf, coils
LINES = [
    ((182, 182), 1.5, 14),  # a prime stage (273 = 3 * 7 * 13): 3920 and 4200 waves in y
    ((182, 182), 1.5, 15),
    ((350, 350), 1.5, 12),  # 525 = 3 * 5^2 * 7: tiles of 1024 threads in x
    ((240, 240), 2.0, 12),  # 480 points, 3840 waves in x: light adjoint, full forward
    ((320, 320), 1.5, 12),  # 480 points, 5120 waves
    ((100, 100), 1.5, 26),  # 256 threads in y: 1976 and 2052 waves
    ((100, 100), 1.5, 27),
    ((48, 48), 1.25, 30),   # 128 threads in y: full tiles
    ((100, 40, 32), 1.25, 2),  # 128 threads in z: 1563 and 2345 light tiles
    ((100, 40, 32), 1.25, 3),
]


@pytest.mark.parametrize("case", LINES, ids=lambda c: "x".join(map(str, c[0])) + "_c%d" % c[2])
def test_same_bits_on_both_sides(case):
    img, osf, C = case
    print("case", case, flush=True)
    torch, pl, k, x = _setup(img, osf, C)
    out = [torch.full_like(x, float("nan")) for _ in range(2)]
    fwd = [torch.full_like(k, float("nan")) for _ in range(2)]
    pl.adjoint(k, out[0], C)
    pl.forward(x, fwd[0], C)
    b = capi.Batch([pl], [C])
    b.adjoint([k], [out[1]])
    b.forward([x], [fwd[1]])
    torch.cuda.synchronize()
    assert torch.isfinite(torch.view_as_real(out[0])).all()
    assert torch.equal(torch.view_as_real(out[0]), torch.view_as_real(out[1]))
    assert torch.equal(torch.view_as_real(fwd[0]), torch.view_as_real(fwd[1]))


@pytest.mark.parametrize("img, osf", [((160, 120), 1.5), ((96, 160), 1.5), ((120, 96), 1.5), ((72, 90), 2.0),
                                      ((128, 150), 1.5), ((128, 128), 1.25), ((64, 64, 16), 1.5), ((48, 40, 120), 1.5)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_bits_do_not_depend_on_the_coils(img, osf):
    """Two coils alone take light passes, among 32 full tiles. (144, 180 and 240
    points: kernels of their own with other stages than by the general order.)"""
    print("case", img, osf, flush=True)
    torch, pl, _, _ = _setup(img, osf, 1)
    pl.set_sens(None, 0)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    rnd = lambda *s: torch.view_as_complex(torch.randn(s + (2,), generator=g, device="cuda"))
    x, k = rnd(32, *reversed(img)), rnd(32, 700)
    fwd = [torch.empty((n, 700), dtype=torch.complex64, device="cuda") for n in (2, 32)]
    adj = [torch.empty((n,) + tuple(reversed(img)), dtype=torch.complex64, device="cuda") for n in (8, 32)]
    for out, n in zip(fwd, (2, 32)):
        pl.forward(x[:n].contiguous(), out, n)
    for out, n in zip(adj, (8, 32)):  # (the spread's groups of eight coils in both)
        pl.adjoint(k[:n].contiguous(), out, n)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(fwd[0]), torch.view_as_real(fwd[1][:2]))
    assert torch.equal(torch.view_as_real(adj[0]), torch.view_as_real(adj[1][:8]))


@pytest.mark.parametrize("case", [((304, 304), 2.0, 32), ((448, 448), 2.0, 32), ((289, 289), 2.0, 32)],
                         ids=lambda c: "x".join(map(str, c[0])) + "_c%d" % c[2])
def test_not_slower_than_full_tiles(case):
    img, osf, C = case
    print("case", case, flush=True)
    torch, pl, k, x = _setup(img, osf, C)
    out, fwd = torch.empty_like(x), torch.empty_like(k)
    b = capi.Batch([pl], [C])

    def alone():
        pl.adjoint(k, out, C)
        pl.forward(x, fwd, C)

    def batch():
        b.adjoint([k], [out])
        b.forward([x], [fwd])

    best = {alone: 1e9, batch: 1e9}
    for _ in range(8):  # in turn; the least of eight blocks of ten
        for f in best:
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            f()
            e[0].record()
            for _ in range(10):
                f()
            e[1].record()
            e[1].synchronize()
            best[f] = min(best[f], e[0].elapsed_time(e[1]))
    print("alone %.1f us, batch %.1f us" % (best[alone] * 100, best[batch] * 100), flush=True)
    assert best[alone] <= best[batch]
