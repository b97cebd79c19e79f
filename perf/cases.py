"""Workloads that a user of this framework runs, for timing and for checking results.

Every case goes through the public entry points: `capi.Plan` (device tensors),
`capi.CGSense`, `capi.Batch` and the drop-in `gpuNUFFT.NUFFTOp` (host arrays).

A case is a dict of plain values:
  kind   "op": adjoint, then forward of one plan; "adjoint" / "forward": one direction;
         "frame": a new trajectory on a kept plan, then the adjoint;
         "cg": a CG-SENSE reconstruction; "batch": `ops` uneven 2-D plans, adjoint and
         forward together; "host": `NUFFTOp.op` and `adj_op` on numpy arrays
  traj   "radial", "spiral" (2-D), "koosh" (3-D) or "stack" (3-D stack of stars)
  nx, ny, nz (0: 2-D)   image size
  osf, kw, sw, linear   oversampling, kernel width, sector width, lookup mode
  coils, sens, dens     coils; coil maps (coil-combined image) and density weights or not
  shots, read           interleaves / spokes (of each partition) and samples of each
"""

import math

import numpy as np
import torch

from gpunufft_amd import capi


def _case(name, kind, traj, nx, ny, nz, osf, kw, sw, linear, coils, sens, dens, shots, read, **more):
    c = dict(kind=kind, traj=traj, nx=nx, ny=ny, nz=nz, osf=osf, kw=kw, sw=sw, linear=linear,
             coils=coils, sens=sens, dens=dens, shots=shots, read=read, **more)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one coil of a 64^2 image (the benchmark's small radial set); launches count
        _case("op2d_64_c1", "op", "radial", 64, 64, 0, 2.0, 3, 8, False, 1, False, True, 64, 128),
        # a slice of a 16-coil radial scan with coil maps, full sampling (the benchmark's 2-D set)
        _case("op2d_256_c16", "op", "radial", 256, 256, 0, 2.0, 3, 8, False, 16, True, True, 402, 512),
        # odd, unequal sides and 1.5-fold oversampling, images of each coil, no density weights
        _case("op2d_301x250_c7", "op", "spiral", 301, 250, 0, 1.5, 3, 8, False, 7, False, False, 24, 2411),
        # wide kernel at low oversampling (the accurate setting), 2-D
        _case("op2d_224_kw5_c12", "op", "spiral", 224, 224, 0, 1.5, 5, 8, False, 12, True, True, 32, 1792),
        # real-time imaging: every frame has its own golden-angle spokes
        _case("frame2d_192_c8", "frame", "radial", 192, 192, 0, 2.0, 3, 8, False, 8, True, True, 55, 384),
        # iterative reconstruction of a slice, ten iterations (the serving loop's request)
        _case("cg2d_240_c12", "cg", "radial", 240, 240, 0, 2.0, 3, 8, False, 12, True, True, 120, 480,
              iterations=10),
        # many slices of different sizes at once
        _case("batch2d_24", "batch", "spiral", 384, 384, 0, 2.0, 3, 16, False, 16, True, True, 48, 4096,
              ops=24, mix=0),
        # the Python drop-in on host arrays with its linear lookup
        _case("host2d_192_c8", "host", "radial", 192, 192, 0, 2.0, 3, 8, True, 8, True, True, 192, 384),
        # the headline: koosh ball 128^3 at 1.5, 8 coils, each direction by itself
        _case("adjoint3d_128_c8", "adjoint", "koosh", 128, 128, 128, 1.5, 3, 8, False, 8, True, True,
              16384, 256),
        _case("forward3d_128_c8", "forward", "koosh", 128, 128, 128, 1.5, 3, 8, False, 8, True, True,
              16384, 256),
        # stack of stars, a flat ragged volume, images of each coil
        _case("op3d_168x160x44_c6", "op", "stack", 168, 160, 44, 1.5, 3, 8, False, 6, False, True, 101, 320),
        # the largest: 160^3 at 2 (a 320^3 grid), undersampled koosh ball (a serving request's shape)
        _case("op3d_160_c8", "op", "koosh", 160, 160, 160, 2.0, 3, 8, False, 8, True, True, 6400, 320),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def side(lo, hi):
        n = log_int(lo, hi)
        return n if rng.random() < 0.25 else max(lo, n // 8 * 8)  # mostly multiples of 8, odd ones among them

    kind = rng.choice(["op", "op", "op", "adjoint", "forward", "frame", "cg", "batch", "host"])
    osf = rng.choice([1.5, 1.5, 2.0, 2.0, 1.25])
    kw = 5 if osf == 1.25 else rng.choice([3, 3, 3, 5])
    sens, dens = rng.random() < 0.7, rng.random() < 0.7
    linear = kind == "host" or rng.random() < 0.15
    three = kind in ("op", "adjoint", "forward") and rng.random() < 0.5
    if kind == "batch":
        return _case(None, "batch", "spiral", 384, 384, 0, 2.0, 3, 16, False, 16, True, True, 48, 4096,
                     ops=rng.randint(4, 24), mix=rng.randint(1, 10 ** 6))
    if three:
        n = side(32, 152)
        coils = rng.randint(1, 8)
        if rng.random() < 0.5:
            shots = min(log_int(max(64, n * n // 8), n * n), 16384)
            return _case(None, kind, "koosh", n, n, n, osf, kw, 8, linear, coils, sens, dens, shots, 2 * n)
        m, nz = side(32, 168), side(16, 64)
        return _case(None, kind, "stack", n, m, nz, osf, kw, 8, linear, coils, sens, dens,
                     log_int(max(16, n // 4), 2 * n), 2 * n)
    n = side(48, 384)
    m = n if rng.random() < 0.6 else side(48, 384)
    coils = 1 if rng.random() < 0.15 else rng.randint(2, 32)
    sw = rng.choice([8, 8, 16])
    if kind == "cg":
        return _case(None, "cg", "radial", n, m, 0, osf, kw, sw, linear, coils, True, True,
                     log_int(max(16, n // 4), n), 2 * n, iterations=rng.randint(5, 10))
    if kind == "host":
        sens, kw, osf = True, 3, rng.choice([1.5, 2.0])
        coils = min(coils, 12)
    traj = "radial" if kind == "frame" else rng.choice(["radial", "spiral"])
    shots, read = (log_int(max(16, n // 8), 2 * n), 2 * n) if traj == "radial" else (
        rng.randint(8, 48), rng.randint(1024, 4096))
    return _case(None, kind, traj, n, m, 0, osf, kw, sw, linear, coils, sens, dens, shots, read)


# ---- inputs -----------------------------------------------------------------


def _trajectory(case, g):
    """float32 [dim][M] in [-0.5, 0.5) on the GPU; the seed turns it."""
    dev = "cuda"
    shots, read = case["shots"], case["read"]
    turn = float(torch.rand((), generator=g, device=dev, dtype=torch.float64)) * 2 * math.pi
    r = torch.arange(read, device=dev, dtype=torch.float64) / read - 0.5
    i = torch.arange(shots, device=dev, dtype=torch.float64)
    if case["traj"] == "koosh":
        z = 1 - 2 * (i + 0.5) / shots
        phi = i * math.pi * (3 - math.sqrt(5)) + turn
        rho = torch.sqrt(torch.clamp(1 - z * z, min=0))
        k = [torch.outer(d, r).reshape(-1) for d in (rho * torch.cos(phi), rho * torch.sin(phi), z)]
    elif case["traj"] == "spiral":
        t = (torch.arange(read, device=dev, dtype=torch.float64) / read) ** 1.5
        turns = max(1.0, case["nx"] / (2.0 * shots))
        a = 2 * math.pi * (turns * t[None, :] + (i / shots)[:, None]) + turn
        k = [(0.5 * t[None, :] * f(a)).reshape(-1) for f in (torch.cos, torch.sin)]
    else:
        a = i * (math.pi / ((1 + math.sqrt(5)) / 2)) + turn
        k = [torch.outer(torch.cos(a), r).reshape(-1), torch.outer(torch.sin(a), r).reshape(-1)]
        if case["traj"] == "stack":
            n = case["nz"]
            z = torch.arange(n, device=dev, dtype=torch.float64) / n - 0.5
            k = [x.repeat(n) for x in k] + [z.repeat_interleave(shots * read)]
    return torch.stack(k).to(torch.float32).clamp_(-0.5, 0.4999999).contiguous()


def _density(traj, power):
    r = torch.sqrt((traj.double() ** 2).sum(0)) ** power
    return (r / r.max()).to(torch.float32).contiguous()


def _shape(case):
    return tuple(n for n in (case["nz"], case["ny"], case["nx"]) if n)


def _coil_maps(case, g):
    """Smooth complex maps [coil][z][y][x] with sum |S|^2 = 1."""
    dev, shape = "cuda", _shape(case)
    at = torch.meshgrid(*[torch.arange(n, device=dev, dtype=torch.float32) / n - 0.5 for n in shape],
                        indexing="ij")
    maps = torch.empty((case["coils"],) + shape, dtype=torch.complex64, device=dev)
    u = torch.rand((case["coils"], 3), generator=g, device=dev, dtype=torch.float64).tolist()
    for c, (a, b, p) in enumerate(u):
        centre = [0.35 * math.sin(2 * math.pi * a), 0.35 * math.cos(2 * math.pi * a)]
        centre = [0.7 * (b - 0.5)] * (len(shape) - 2) + centre
        d2 = sum((x - x0) ** 2 for x, x0 in zip(at, centre))
        maps[c] = torch.exp(-d2 / 0.18) * complex(math.cos(2 * math.pi * p), math.sin(2 * math.pi * p))
    return maps / torch.sqrt((maps.abs() ** 2).sum(0))


def _noise(shape, g):
    return torch.view_as_complex(torch.randn(tuple(shape) + (2,), generator=g, device="cuda"))


def _kspace(case, traj, g):
    """Complex noise under the decay that an image's spectrum has."""
    fall = 1 / (1 + 30 * torch.sqrt((traj ** 2).sum(0)))
    return (_noise((case["coils"], traj.shape[1]), g) * fall).contiguous()


def _image(case, channels, g):
    """A few soft blobs over a little noise, [channel][z][y][x]."""
    shape = _shape(case)
    at = torch.meshgrid(*[torch.arange(n, device="cuda", dtype=torch.float32) / n - 0.5 for n in shape],
                        indexing="ij")
    img = 0.05 * _noise((channels,) + shape, g)
    u = torch.rand((channels, 3, 5), generator=g, device="cuda", dtype=torch.float64).tolist()
    for c in range(channels):
        for x0, x1, x2, w, p in u[c]:
            d2 = sum((x - 0.6 * (o - 0.5)) ** 2 for x, o in zip(at, (x0, x1, x2)))
            img[c] += torch.exp(-d2 / (0.01 + 0.05 * w)) * complex(math.cos(6.28 * p), math.sin(6.28 * p))
    return img.contiguous()


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    kind, sens = case["kind"], case["sens"]
    traj = _trajectory(case, g)
    s = dict(traj=traj, dens=_density(traj, 1 if len(traj) == 2 else 2) if case["dens"] else None,
             sens=_coil_maps(case, g) if sens else None)
    if kind != "forward":
        s["kdata"] = _kspace(case, traj, g)
    if kind in ("op", "forward", "batch", "host"):
        s["img"] = _image(case, 1 if sens else case["coils"], g)
    return s


def _batch_cases(case):
    """The uneven plans of a batch: sides, interleaves, lengths and coils up to the case's."""
    r = np.random.default_rng(case["mix"])  # the mix belongs to the case, not to the seed
    got = []
    for _ in range(case["ops"]):
        n = int(r.choice([96, 128, 192, 256, 320, 384]))
        got.append(dict(case, kind="op", nx=min(n, case["nx"]), ny=min(n, case["ny"]),
                        coils=int(r.integers(4, case["coils"] + 1)),
                        shots=int(r.integers(8, case["shots"] + 1)),
                        read=int(r.integers(1024, case["read"] + 1))))
    return got


# ---- the program ------------------------------------------------------------


def _plan(case, s):
    dims = [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] else [])
    p = capi.Plan(dims, case["kw"], case["sw"], case["osf"],
                  capi.LOOKUP_LINEAR if case["linear"] else capi.LOOKUP_NEAREST)
    p.set_trajectory(s["traj"], s["dens"])
    if s["sens"] is not None:
        p.set_sens(s["sens"], case["coils"])
    return p


def _buffers(case, s):
    shape, m = _shape(case), s["traj"].shape[1]
    return (torch.empty(((1 if case["sens"] else case["coils"]),) + shape, dtype=torch.complex64, device="cuda"),
            torch.empty((case["coils"], m), dtype=torch.complex64, device="cuda"))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        cases = _batch_cases(case)
        parts = [_inputs(c, int(seed) * 1009 + j) for j, c in enumerate(cases)]
        plans = [_plan(c, s) for c, s in zip(cases, parts)]
        out = [_buffers(c, s) for c, s in zip(cases, parts)]
        batch = capi.Batch(plans, [c["coils"] for c in cases])
        return dict(case=case, batch=batch, plans=plans, kdata=[s["kdata"] for s in parts],
                    img=[s["img"] for s in parts], x=[o[0] for o in out], k=[o[1] for o in out])
    s = _inputs(case, seed)
    if kind == "host":
        from gpunufft_amd.gpuNUFFT import NUFFTOp

        dims = [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] else [])
        h = {k: v.cpu().numpy() for k, v in s.items() if v is not None}
        op = NUFFTOp(h["traj"], np.array(dims, np.int32), case["coils"], h["sens"],
                     h.get("dens", np.zeros(0, np.float32)), case["kw"], case["sw"], case["osf"], True)
        return dict(case=case, op=op, img=h["img"], kdata=h["kdata"])
    x, k = _buffers(case, s)
    state = dict(case=case, plan=_plan(case, s), x=x, k=k, coils=case["coils"], **s)
    if kind == "cg":
        state["cg"] = capi.CGSense(state["plan"], case["coils"], 1e-3)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].adjoint(state["kdata"], state["x"])
        state["batch"].forward(state["img"], state["k"])
        return {"x": state["x"], "k": state["k"]}
    if kind == "host":
        return {"k": state["op"].op(state["img"]), "x": state["op"].adj_op(state["kdata"])}
    if kind == "cg":
        return {"x": state["cg"].solve(state["kdata"], state["x"], case["iterations"])}
    plan, got = state["plan"], {}
    if kind == "frame":
        plan.set_trajectory(state["traj"], state["dens"])
    if kind in ("op", "adjoint", "frame"):
        got["x"] = plan.adjoint(state["kdata"], state["x"], state["coils"])
    if kind in ("op", "forward"):
        got["k"] = plan.forward(state["img"], state["k"], state["coils"])
    return got


def _samples(case):
    return case["shots"] * case["read"] * (case["nz"] if case["traj"] == "stack" else 1)


def work(case):
    """Samples, trajectory, weights, maps and image once each; taps and FFTs."""
    if case["kind"] == "batch":
        w = [work(c) for c in _batch_cases(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    shape = _shape(case)
    d, m, c = len(shape), _samples(case), case["coils"]
    ni = math.prod(shape)
    ng = math.prod(int(n * case["osf"]) for n in shape)
    one = 8 * m * c + 4 * d * m + (4 * m if case["dens"] else 0) + 8 * ni * (1 + c if case["sens"] else c)
    flop = c * (4 * m * case["kw"] ** d + 5 * ng * math.log2(ng))
    passes = {"op": 2, "host": 2, "cg": 1 + 2 * case.get("iterations", 0)}.get(case["kind"], 1)
    return {"bytes": one * passes, "flops": flop * passes}


# ---- the same in 64 bits ------------------------------------------------------


def _table(case):
    """Kaiser-Bessel table over r^2 / radius^2; its length follows the oversampling in float32."""
    osf, kw = np.float32(case["osf"]), case["kw"]
    if case["linear"]:
        per = math.floor(math.sqrt(0.37 / float(osf * osf * np.float32(0.0001))))
    else:
        per = math.floor(np.float32(0.91) / (osf * np.float32(0.001)))
    n = int(per * kw * 0.5)
    beta = math.pi * math.sqrt((kw / case["osf"] * (case["osf"] - 0.5)) ** 2 - 0.8)
    r2 = np.arange(n) / (n - 1)
    t = np.i0(beta * np.sqrt(np.maximum(0.0, 1 - r2))) / np.i0(beta)
    t[0], t[-1] = 1.0, 0.0
    return torch.from_numpy(t).cuda()


def _taps(case, pos, size, most, table, sw):
    """Grid indices and float64 weights [kw + 1][M] of positions along one axis. Which entry of
    the table a tap takes is settled in float32, as part of the operator's definition."""
    f = torch.float32
    kw, n = case["kw"], len(table)
    pad = sw + 2 * (kw // 2)
    off, half = pad // 2, kw / 2.0
    sector = torch.floor(torch.floor((pos * size).double() + 0.5 * size + 0.5) / sw)
    centre = sector.clamp(0, math.ceil(size / sw) - 1) * sw + sw // 2
    cf = centre.to(f)
    u = (pos * size) + 0.5 * size - cf + off
    lo = torch.ceil(u - half).clamp(min=0)
    lo = torch.where(lo >= pad - 1, torch.full_like(lo, float(int(pad - 1 - 2 * half))), lo)
    hi = torch.floor(u + half).clamp(0, pad - 1)
    radius2 = (half / most) ** 2
    whole = torch.full_like(pos, size)  # a true division: by a number it would be a product
    idx, wts = [], []
    for t in range(kw + 1):
        i = lo + t
        d = ((i + cf - off) / whole - 0.5 - pos) * float(np.float32(size) / np.float32(most))
        d = d * d
        if case["linear"]:
            x = d * float(np.float32(1.0 / radius2)) * float(n) - 0.5
            a = torch.round((x - torch.floor(x)) * 256).double() / 256
            i0 = torch.floor(x).long()
            w = (1 - a) * table[i0.clamp(0, n - 1)] + a * table[(i0 + 1).clamp(0, n - 1)]
        else:
            e = torch.floor((d * float(np.float32((n - 1) / radius2))).double() + 0.5).long()
            w = table[e.clamp(max=n - 1)] * (d < float(np.float32(radius2)))
        idx.append((centre - off + i.double()).long() % size)
        wts.append(w * (i <= hi))
    return idx, wts


class _Exact:
    def __init__(self, case, s):
        self.case, self.sens = case, s["sens"]
        self.N = _shape(case)
        self.G = tuple(int(n * np.float32(case["osf"])) for n in self.N)
        self.ng, ni = math.prod(self.G), math.prod(self.N)
        table, most, d = _table(case), max(self.G), len(self.N)
        self.root = s["dens"].double().sqrt() if s["dens"] is not None else None
        self.taps = [_taps(case, s["traj"][d - 1 - a], self.G[a], most, table, case["sw"]) for a in range(d)]
        self.taps = [[(i, w) for i, w in zip(*t) if float(w.abs().max()) > 0] for t in self.taps]
        # image position of pixel x: crop + centre; 1 / |transform of the kernel at the origin|
        self.at, deapo = [], torch.full((1,) * d, math.sqrt(self.ng / ni), dtype=torch.float64, device="cuda")
        zero = torch.zeros(1, dtype=torch.float32, device="cuda")
        for a, (n, size) in enumerate(zip(self.N, self.G)):
            crop = int(np.float32(n) * (np.float32(case["osf"]) - np.float32(1)) / np.float32(2))
            x = torch.arange(n, device="cuda") + crop
            self.at.append(x)
            idx, wts = _taps(case, zero, size, most, table, 8)
            m = (x + size // 2) % size
            f = sum(w * torch.exp(2j * math.pi * ((((i - size // 2) % size) * m) % size).double() / size)
                    for i, w in zip(idx, wts))
            deapo = deapo / f.abs().reshape([-1 if b == a else 1 for b in range(d)])
        self.deapo = deapo

    def _each_tap(self, a=0, j=None, v=None):
        for i, w in self.taps[a]:
            jj = i if j is None else j * self.G[a] + i
            vv = w if v is None else v * w
            if a + 1 < len(self.G):
                yield from self._each_tap(a + 1, jj, vv)
            else:
                yield jj, vv

    def adjoint(self, kdata):
        c = kdata.shape[0]
        val = kdata.to(torch.complex128)
        if self.root is not None:
            val = val * self.root
        val = torch.view_as_real(val.T.contiguous()).reshape(-1, 2 * c)  # [M][coil re, im]
        grid = torch.zeros((self.ng, 2 * c), dtype=torch.float64, device="cuda")
        for j, w in self._each_tap():
            grid.index_add_(0, j, val * w[:, None])
        dims = tuple(range(len(self.G)))
        out = None if self.sens is not None else torch.empty((c,) + self.N, dtype=torch.complex128, device="cuda")
        for k in range(c):
            x = torch.view_as_complex(grid[:, 2 * k:2 * k + 2].contiguous()).reshape(self.G)
            x = torch.roll(x, [-(n // 2) for n in self.G], dims)
            x = torch.fft.ifftn(x, norm="forward")
            for a, (at, n) in enumerate(zip(self.at, self.G)):
                x = x.index_select(a, (at + n // 2) % n)
            x = x * (self.deapo / math.sqrt(self.ng))
            if self.sens is None:
                out[k] = x
            else:
                x = x * self.sens[k].to(torch.complex128).conj()
                out = x if out is None else out + x
        return out if self.sens is None else out[None]

    def forward(self, img):
        c = self.case["coils"]
        m = self.taps[0][0][0].numel()
        grid = torch.empty((self.ng, 2 * c), dtype=torch.float64, device="cuda")
        for k in range(c):
            x = img[0 if self.sens is not None else k].to(torch.complex128) * self.deapo
            if self.sens is not None:
                x = x * self.sens[k].to(torch.complex128)
            full = torch.zeros(self.G, dtype=torch.complex128, device="cuda")
            where = torch.meshgrid(*[(at - n // 2) % n for at, n in zip(self.at, self.G)], indexing="ij")
            full[where] = x
            full = torch.fft.fftn(full)
            full = torch.roll(full, [-((n + 1) // 2) for n in self.G], tuple(range(len(self.G))))
            grid[:, 2 * k:2 * k + 2] = torch.view_as_real(full).reshape(-1, 2)
        val = torch.zeros((m, 2 * c), dtype=torch.float64, device="cuda")
        for j, w in self._each_tap():
            val += grid[j] * w[:, None]
        val = torch.view_as_complex(val.reshape(m, c, 2)).T / math.sqrt(self.ng)
        return (val * self.root if self.root is not None else val).contiguous()


def _exact_cg(op, case, kdata):
    def dot(a, b):
        return float((a.conj() * b).sum().real)

    r = op.adjoint(kdata)
    x, p, rr = torch.zeros_like(r), r, dot(r, r)
    for _ in range(case["iterations"]):
        q = op.adjoint(op.forward(p)) + float(np.float32(1e-3)) * p
        a = rr / dot(p, q)
        x, r = x + a * p, r - a * q
        new = dot(r, r)
        p, rr = r + (new / rr) * p, new
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        got = [exact(c, int(seed) * 1009 + j) for j, c in enumerate(_batch_cases(case))]
        return {"x": [g["x"] for g in got], "k": [g["k"] for g in got]}
    s = _inputs(case, seed)
    op, got = _Exact(case, s), {}
    if kind == "cg":
        return {"x": _exact_cg(op, case, s["kdata"])}
    if kind in ("op", "adjoint", "frame", "host"):
        got["x"] = op.adjoint(s["kdata"])
    if kind in ("op", "forward", "host"):
        got["k"] = op.forward(s["img"])
    return got
