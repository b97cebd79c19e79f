"""Admission's memory estimate against what a request takes.

On the CPU: lower and upper bounds put together from the sizes of the buffers that
every request has. On the GPU: the memory gone from the device once a request is
active is within the estimate, and the estimate within twice that (and 96 MiB of
allocation granularity).
"""

import numpy as np
import pytest

from gpunufft_amd import serve
from gpunufft_amd import workloads as W


def _request(dims, C, M, osf, kw=3, sw=8, centre=False):
    rng = np.random.default_rng(M)
    d = len(dims)
    traj = rng.normal(0, 0.08, (d, M)) if centre else rng.uniform(-0.5, 0.4999, (d, M))
    traj = np.clip(traj, -0.5, 0.4999).astype(np.float32)
    return serve.Request(rid=0, arrival=0.0, img_dims=dims, traj=traj, dens=np.ones(M, np.float32),
                         sens=np.ones((C,) + tuple(dims[::-1]), np.complex64), kdata=np.ones((C, M), np.complex64),
                         osf=osf, kernel_width=kw, sector_width=sw, iterations=1)


def test_dense_small_grid_is_not_underestimated():
    # 4 M samples on a 96^3 grid: per sample 48 bytes of taps, 4 of its sorted
    # position, 12 + 8 of trajectory and density tables, 4 of square roots... at
    # least one list entry, the caller's arrays and the solver's k-space
    M = 4 << 20
    r = _request((64, 64, 64), 1, M, 1.5)
    per_sample = 48 + 4 + 12 + 4 + 4 + 8 + 4 + 16 + 8 + 8
    assert r.device_bytes() >= M * per_sample + 8 * 96 ** 3


def test_large_request_is_not_overestimated():
    # 152^3 at osf 2, 8 coils, 1.76 M samples: the work grid, the FFT's intermediate
    # (half of it), coil maps twice, solver vectors and 200 bytes a sample
    N, C, M = 152, 8, 5776 * 304
    r = _request((N, N, N), 1, 1000, 2.0)
    r.traj, r.sens = np.broadcast_to(np.float32(0), (3, M)), np.broadcast_to(np.complex64(0), (C, N, N, N))
    need = C * 8 * ((2 * N) ** 3 * 1.5 + 2 * N ** 3 + 2 * M) + 7 * 8 * N ** 3 + 200 * M
    assert need <= 1.1 * r.device_bytes() and r.device_bytes() <= 1.25 * need


def test_serving_mix_is_within_the_device():
    for r in serve.serving_mix(8, seed=3):
        assert 0 < r.device_bytes() < 16 << 30


@pytest.mark.gpu
@pytest.mark.parametrize("args", [
    dict(dims=(64, 64, 64), C=1, M=4 << 20, osf=1.5),
    dict(dims=(64, 64, 64), C=2, M=1 << 20, osf=1.5, centre=True),
    dict(dims=(120, 120, 120), C=8, M=1 << 20, osf=2.0),
    dict(dims=(384, 384), C=32, M=1 << 20, osf=2.0),
    dict(dims=(256, 256), C=16, M=200000, osf=1.5, kw=5),
    dict(dims=(350, 301), C=12, M=300000, osf=1.5, centre=True),
    dict(dims=(50, 50, 50), C=8, M=300000, osf=1.5),
], ids=lambda a: "x".join(map(str, a["dims"])) + "_c%d" % a["C"])
def test_estimate_covers_what_is_taken(args):
    import torch
    print("case", args, flush=True)
    r = _request(**args)
    s = serve.Server(slots=1)
    warm = s._start(_request((16, 16), 1, 100, 2.0), 0)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    a = s._start(r, 0)
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    est = r.device_bytes()
    print("taken %.1f MB, estimate %.1f MB" % (taken / 1e6, est / 1e6), flush=True)
    for x in (a, warm):
        x["cg"].close()
        x["plan"].close()
    assert taken <= est + (96 << 20)
    assert est <= 2 * taken + (96 << 20)
