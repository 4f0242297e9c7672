"""Workloads of the backprojector as its users run them: the cases that timings are taken on.

Every capture is synthetic: relay wall z = 0, scan grids over [-1, 1]^2 m, laser and SPAD origins
at ORIGIN, a hidden volume of about 1 m across 0.3 m behind the wall, time axis of 4.096 m in T
bins.  The hidden scene is a few bright points and two patches facing the wall; samples are photon
counts (Poisson draws of the 1/r^4 falloff plus a sparse background), or real values where a case
says so (counts minus the background, times a gain: what a calibrated capture holds).

kind        what a user's program does
oneshot     `nlosbpy.backproject` on host arrays (the reference module's main call)
window      the same with use_cpu=True: the reference CPU path's semantics
phasor      `nlosbpy.phasor` on host arrays (complex volume)
plan        a `Plan` kept for one capture: execute, then read the volume
octree      an octree `Plan` with the shipped proposal net at its shipped operating point
batch       a `Batch` of captures of different sizes: execute, then read every volume
scan        confocal | exhaustive (every laser with every SPAD) | pairs (a list without structure)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from backprojector_amd import core, nlosbpy, proposals

ORIGIN = np.array([0.0, -1.0, 0.5], np.float32)
VOLUME_POSITION = np.array([0.0, 0.0, 0.8], np.float32)
VOLUME_SIZE = np.array([1.0, 1.0, 1.0], np.float32)
RANGE = 4.096          # metres of path that the time axis covers
CYCLES = 4             # wave cycles of a phasor pulse


def listed():
    return [
        # the command line's default volume (32^3) from a small scan: the smallest call
        dict(name="oneshot_32", kind="oneshot", scan="confocal", sx=32, sy=32, T=1024, nx=32, ny=32, nz=32,
             samples="counts"),
        # a scan and a volume with no round size, kept as a plan (previews while a rig is set up)
        dict(name="plan_ragged", kind="plan", scan="confocal", sx=37, sy=53, T=1500, nx=45, ny=61, nz=38,
             samples="counts", storage="f32"),
        # the standard reconstruction: 128 x 128 confocal photon counts into 128^3
        dict(name="plan_128", kind="plan", scan="confocal", sx=128, sy=128, T=4096, nx=128, ny=128, nz=128,
             samples="counts", storage="f32"),
        # a calibrated (real-valued) capture
        dict(name="plan_real", kind="plan", scan="confocal", sx=96, sy=96, T=4096, nx=128, ny=120, nz=100,
             samples="real", storage="f32"),
        # real values in 16-bit storage
        dict(name="plan_bf16", kind="plan", scan="confocal", sx=64, sy=64, T=2048, nx=96, ny=96, nz=96,
             samples="real", storage="bf16"),
        # the largest volume: 256^3
        dict(name="plan_256", kind="plan", scan="confocal", sx=128, sy=128, T=4096, nx=256, ny=256, nz=256,
             samples="counts", storage="f32"),
        # 16 x 16 lasers with 16 x 16 SPADs
        dict(name="plan_exhaustive", kind="plan", scan="exhaustive", sx=16, sy=16, T=4096, nx=64, ny=64, nz=64,
             samples="counts", storage="f32"),
        # laser and SPAD spots in no order (the pairs of an exhaustive scan, shuffled)
        dict(name="plan_pairs", kind="plan", scan="pairs", sx=12, sy=12, T=2048, nx=48, ny=48, nz=48,
             samples="counts", storage="f32"),
        # one phasor-field reconstruction from host arrays, 4 cm wavelength
        dict(name="phasor_64", kind="phasor", scan="confocal", sx=64, sy=64, T=2048, nx=64, ny=64, nz=64,
             samples="counts", wavelength=0.04),
        # the reference CPU path's semantics (its default when no GPU is asked for)
        dict(name="window_96", kind="window", scan="confocal", sx=96, sy=96, T=2048, nx=96, ny=96, nz=96,
             samples="counts"),
        # coarse-to-fine reconstruction of 256^3 with the learned proposals
        dict(name="octree_256", kind="octree", scan="confocal", sx=128, sy=128, T=4096, nx=256, ny=256, nz=256,
             samples="counts"),
        # captures of many sizes served together
        dict(name="batch_16", kind="batch", captures=16, updates=1.2e10, sx=128, T=4096, nx=96),
    ]


# The most voxel-pair updates of a drawn case of each kind: a drawn case stays below the listed ones.
DRAW_KINDS = {("oneshot", "confocal"): 1.0e10, ("plan", "confocal"): 3.4e10, ("plan", "exhaustive"): 8.0e9,
              ("plan", "pairs"): 2.0e9, ("phasor", "confocal"): 2.0e9, ("window", "confocal"): 6.0e9,
              ("oneshot", "exhaustive"): 4.0e9, ("batch", ""): 1.0e10}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind, scan = rng.choice(sorted(DRAW_KINDS))
    most = DRAW_KINDS[kind, scan]
    if kind == "batch":
        return dict(kind=kind, captures=rng.randint(4, 20), updates=_log_int(rng, 1e9, most), sx=_log_int(rng, 48, 128),
                    T=rng.randint(1024, 4096), nx=_log_int(rng, 32, 96))
    lo, hi = (16, 128) if scan == "confocal" else (5, 16)
    c = dict(kind=kind, scan=scan, sx=_log_int(rng, lo, hi), sy=_log_int(rng, lo, hi), T=_log_int(rng, 512, 4096),
             nx=_log_int(rng, 16, 128), ny=_log_int(rng, 16, 128), nz=_log_int(rng, 16, 128),
             samples=rng.choice(["counts", "counts", "real"]))
    while _pairs_of(c) * c["nx"] * c["ny"] * c["nz"] > most:
        axis = rng.choice(["nx", "ny", "nz"])
        c[axis] = max(16, int(c[axis] * 0.9))
    if kind == "plan":
        c["storage"] = rng.choice(["f32", "f32", "f16", "bf16"])
    if kind == "phasor":
        c["wavelength"] = rng.choice([0.04, 0.05, 0.06])
    return c


def _pairs_of(case):
    return case["sx"] * case["sy"] * (1 if case["scan"] == "confocal" else case["sx"] * case["sy"])


# ------------------------------------------------------------------ captures
def _grid(nx, ny):
    gx, gy = np.linspace(-1.0, 1.0, nx), np.linspace(-1.0, 1.0, ny)
    X, Y = np.meshgrid(gx, gy, indexing="ij")
    return np.stack([X, Y, np.zeros_like(X)], -1).astype(np.float32)


def _dist64(a, b):
    """The reference's host distance: float differences, double squares, sum and root."""
    d = (np.asarray(a, np.float32) - np.asarray(b, np.float32)).astype(np.float64)
    return np.sqrt(d[..., 0] ** 2 + d[..., 1] ** 2 + d[..., 2] ** 2)


def _geometry(case):
    """(camera grid, laser grid, laser points [P,3], camera points [P,3], wall distances [P] x 2)."""
    if case["scan"] == "confocal":
        cg = _grid(case["sx"], case["sy"])
        cp = cg.reshape(-1, 3)
        w = _dist64(cp, ORIGIN).astype(np.float32)
        return cg, cg, cp, cp, w, w
    g = _grid(case["sx"], case["sy"])
    pts = g.reshape(-1, 3)
    w = _dist64(pts, ORIGIN).astype(np.float32)
    n = len(pts)
    return g, g, np.repeat(pts, n, 0), np.tile(pts, (n, 1)), np.repeat(w, n), np.tile(w, n)


def _samples(lp, cp, lw, cw, T, seed, real):
    """[P][T] float32 samples on the host: photon counts, or real values made of them."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed) * 1000003 + 17)
    r = np.random.default_rng(int(seed) + 1000)
    pts = r.uniform((-0.4, -0.4, 0.5), (0.4, 0.4, 1.2), (8, 3))
    parts, weight, facing = [pts], [np.full(8, 1e-3)], [np.zeros(8)]
    for _ in range(2):
        k, size = 24, 0.3
        u = (np.arange(k) + 0.5) / k * size - size / 2
        c = r.uniform(-0.35, 0.35, 2)
        X, Y = np.meshgrid(c[0] + u, c[1] + u, indexing="ij")
        parts.append(np.stack([X.ravel(), Y.ravel(), np.full(k * k, r.uniform(0.6, 1.1))], -1))
        weight.append(np.full(k * k, (size / k) ** 2))
        facing.append(np.ones(k * k))
    q = torch.tensor(np.concatenate(parts), dtype=torch.float64, device=dev)
    a = torch.tensor(np.concatenate(weight), dtype=torch.float64, device=dev)
    f = torch.tensor(np.concatenate(facing), dtype=torch.bool, device=dev)
    L, C = (torch.tensor(x, dtype=torch.float64, device=dev) for x in (lp, cp))
    wall = torch.tensor(np.asarray(lw, np.float64) + cw, device=dev)
    P = len(lp)
    out = torch.empty((P, T), dtype=torch.float32, device=dev)
    step = max(1, min(4096, (1 << 26) // T))
    for p in range(0, P, step):
        e = min(P, p + step)
        dl = (L[p:e, None] - q).norm(dim=-1)
        ds = (C[p:e, None] - q).norm(dim=-1)
        b = ((wall[p:e, None] + dl + ds) * (T / RANGE)).floor().long()
        cos = torch.where(f, (q[:, 2] / dl) * (q[:, 2] / ds), 1.0)
        lam = 2.0e4 * a * cos / (dl * ds) ** 2
        hits = torch.poisson(lam.float(), generator=gen).to(torch.int32)
        hits = torch.where((b >= 0) & (b < T), hits, 0)
        rows = torch.poisson(torch.full((e - p, T), 0.02, device=dev), generator=gen).to(torch.int32)
        rows.scatter_add_(1, b.clamp(0, T - 1), hits)
        out[p:e] = (rows.float() - 0.02) * 0.731 if real else rows.float()
    return out.cpu().numpy()


def _capture(case, seed):
    cg, lg, lp, cp, lw, cw = _geometry(case)
    H = _samples(lp, cp, lw, cw, case["T"], seed, case["samples"] == "real")
    pairs = np.zeros(len(lp), core.PAIR_DTYPE)
    pairs["camera_point"], pairs["laser_point"], pairs["camera_wall"], pairs["laser_wall"] = cp, lp, cw, lw
    if case["scan"] == "pairs":
        perm = np.random.default_rng(int(seed) + 7).permutation(len(pairs))
        H, pairs = H[perm], pairs[perm]
    return H, pairs, cg, lg


def _volume_grid(case):
    """Voxel (0, 0, 0) and the 3 x 3 increments of the single-tap grid: spacing size / (N - 1)."""
    N = (case["nx"], case["ny"], case["nz"])
    zero = VOLUME_POSITION - VOLUME_SIZE / np.float32(2)
    inc = np.diag([VOLUME_SIZE[k] / np.float32(N[k] - 1) for k in range(3)]).astype(np.float32).ravel()
    return N, zero, inc


def _batch_members(case, seed):
    """Cases of a batch's captures: wall sides, bins and volumes of mixed sizes (drawn from the case's own
    sizes, not from the seed: a service's mix of sizes stays while its captures change)."""
    r = np.random.default_rng(1004 + case["captures"])
    out = []
    for _ in range(case["captures"]):
        side = max(16, int(case["sx"] * r.choice([0.125, 0.25, 0.5, 0.75, 1.0])))
        n = max(16, int(case["nx"] * r.choice([0.25, 0.33, 0.5, 0.75, 1.0])))
        out.append(dict(kind="plan", scan="confocal", sx=side, sy=side, T=max(512, int(case["T"] * r.choice([0.25, 0.5, 1.0]))),
                        nx=n, ny=n, nz=n, samples="counts"))
    while sum(_pairs_of(c) * c["nx"] ** 3 for c in out) > case["updates"]:
        big = max(out, key=lambda c: _pairs_of(c) * c["nx"] ** 3)
        big["sx"] = big["sy"] = max(16, int(big["sx"] * 0.8))
        big["nx"] = big["ny"] = big["nz"] = max(16, int(big["nx"] * 0.9))
    return out


# ------------------------------------------------------------------ the cases
def prepare(case, seed):
    kind, dT = case["kind"], RANGE / case["T"]
    if kind == "batch":
        args = []
        for i, m in enumerate(_batch_members(case, seed)):
            H, pairs, _, _ = _capture(m, 100 * seed + i)
            args.append((H, pairs, *_volume_grid(m), 0.0, RANGE / m["T"]))
        return dict(kind=kind, batch=core.Batch(args), count=len(args))
    H, pairs, cg, lg = _capture(case, seed)
    N, zero, inc = _volume_grid(case)
    if kind == "plan":
        return dict(kind=kind, plan=core.Plan(H, pairs, N, zero, inc, 0.0, dT, storage=case["storage"]))
    if kind == "octree":
        plan = core.Plan.octree(H, pairs, N, zero, inc, 0.0, dT, levels=4, threshold=0.25)
        net, meta = proposals.load()
        proposals.apply_operating_point(plan, net, 0.25, meta["proposal_threshold"])
        return dict(kind=kind, plan=plan, net=net)
    confocal = case["scan"] == "confocal"
    shape = cg.shape[:2] + (case["T"],) if confocal else lg.shape[:2] + cg.shape[:2] + (case["T"],)
    return dict(kind=kind, wavelength=case.get("wavelength"),
                args=(H.reshape(shape), cg, lg, ORIGIN, ORIGIN, 0.0, dT, confocal, VOLUME_POSITION, VOLUME_SIZE, N))


def run(state):
    kind = state["kind"]
    if kind in ("plan", "octree"):
        state["plan"].execute()
        return state["plan"].volume()
    if kind == "batch":
        state["batch"].execute()
        return [state["batch"].volume(i) for i in range(state["count"])]
    if kind == "phasor":
        return nlosbpy.phasor(*state["args"], state["wavelength"], assume_row_major=True)
    return nlosbpy.backproject(*state["args"], (0.0, 0.0, 0.0), assume_row_major=True, use_cpu=kind == "window")


def work(case):
    """Samples read once, pair records read once, the volume written once; per voxel-pair update the squared
    distance (2 operations: the x and y terms belong to the column), its root, the quotient (2) and the add,
    twice the distance where laser and SPAD differ, a complex add for a phasor, two edges for a window."""
    if case["kind"] == "batch":
        parts = [work(m) for m in _batch_members(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    P, V = _pairs_of(case), case["nx"] * case["ny"] * case["nz"]
    cplx = case["kind"] == "phasor"
    b = P * case["T"] * 4 + P * 32 + V * (8 if cplx else 4)
    per = 6 + (3 if case["scan"] != "confocal" else 0) + (1 if cplx else 0) + (3 if case["kind"] == "window" else 0)
    if case["kind"] == "octree":       # the exact voxels are about a twentieth of the volume
        return {"bytes": b, "flops": P * V * per / 20}
    fir = 4.0 * P * case["T"] * int(CYCLES * case["wavelength"] / (RANGE / case["T"])) if cplx else 0.0
    return {"bytes": b, "flops": P * V * per + fir}


# ------------------------------------------------------------------ values in 64 bits
def _f32(x):
    """Rounds a float64 tensor to float32 and back (a root or a quotient rounded this way is the correctly
    rounded float32 one)."""
    return x.float().double()


def _dist32(pts, v):
    """The float32 distances [P, V] of the single-tap formula, as float64 values."""
    d = [_f32(pts[:, None, k] - v[None, :, k]) for k in range(3)]
    s = _f32(_f32(_f32(d[0] * d[0]) + _f32(d[1] * d[1])) + _f32(d[2] * d[2]))
    return _f32(s.sqrt())


def _positions(N, zero, inc):
    """Voxel positions [V, 3] of the single-tap grid: every operation rounded to float32."""
    z, m = zero.astype(np.float32), inc.astype(np.float32).reshape(3, 3)
    i = np.meshgrid(*[np.arange(n, dtype=np.float32) for n in N], indexing="ij")
    v = [((z[k] + m[0, k] * i[0]) + m[1, k] * i[1]) + m[2, k] * i[2] for k in range(3)]
    return torch.tensor(np.stack(v, -1).reshape(-1, 3).astype(np.float64), device="cuda")


def _single_tap(H, pairs, N, zero, inc, t0, dT):
    """Volume of samples H [P][T] (float64 or complex128) by the float32 path-length formula, summed in 64 bits."""
    dev = torch.device("cuda")
    v = _positions(N, zero, inc)
    lp, cp = (torch.tensor(pairs[k].astype(np.float64), device=dev) for k in ("laser_point", "camera_point"))
    lw, cw = (torch.tensor(pairs[k].astype(np.float64), device=dev) for k in ("laser_wall", "camera_wall"))
    same = bool(np.array_equal(pairs["laser_point"], pairs["camera_point"]))
    t0, dT = float(np.float32(t0)), float(np.float32(dT))
    H = torch.as_tensor(H, device=dev)
    T = H.shape[1]
    out = torch.zeros(len(v), dtype=torch.complex128 if H.is_complex() else torch.float64, device=dev)
    step = max(1, (1 << 25) // len(v))
    for p in range(0, len(lp), step):
        e = min(len(lp), p + step)
        d1 = _dist32(lp[p:e], v)
        d2 = d1 if same else _dist32(cp[p:e], v)
        total = _f32(_f32(_f32(lw[p:e, None] + d1) + d2) + cw[p:e, None])
        q = _f32(_f32(total - t0) / dT)
        b = torch.where(q >= 0, torch.floor(q + 0.5), torch.ceil(q - 0.5))
        inside = (b >= 0) & (b < T)
        x = torch.gather(H[p:e], 1, torch.where(inside, b, 0.0).long())
        out += torch.where(inside, x.to(out.dtype), 0).sum(0)
    return out.reshape(tuple(N)).cpu()


def _time_limits(cg, lg, dT):
    """First and last bin of the reference pipeline's chunk, in float32 (t0 = 0)."""
    las = lg[[0, 0, -1, -1], [0, -1, 0, -1]]
    # the reference takes the camera corners from the transposed grid: entry (k, y) of column c
    cam = np.stack([[cg[k, y, c] for k in range(3)] for c in (0, 2) for y in (0, -1)])
    lower = VOLUME_POSITION - VOLUME_SIZE / np.float32(2)
    vol = np.stack([[lower[k] + np.float32(1.0 if m & (1 << (2 - k)) else 0.0) * VOLUME_SIZE[k] for k in range(3)]
                    for m in range(8)]).astype(np.float32)
    lo = hi = None
    for a, b in ((ORIGIN[None], las), (ORIGIN[None], cam), (vol, las), (vol, cam)):
        d = _dist64(a[:, None], b[None]).astype(np.float32)
        lo = d.min() if lo is None else lo + d.min()
        hi = d.max() if hi is None else hi + d.max()
    dT = np.float32(dT)
    return lo / dT - np.float32(100), hi / dT + np.float32(100)


def _chunk(H, lo, hi):
    """Samples [P][Tc] of bins floor(lo) .. ceil(hi), zero where the capture has none."""
    a, b, T = int(math.floor(lo)), int(math.ceil(hi)), H.shape[1]
    out = torch.zeros((H.shape[0], b - a), dtype=torch.float64, device="cuda")
    f, t = max(a, 0), min(b, T)
    if t > f and (f - a) + (t - f) <= b - a:
        out[:, f - a:t - a] = torch.as_tensor(H[:, f:t], device="cuda").double()
    return out


def _phasor_rows(H, wavelength, dT):
    """The phasor pulse along the rows in 64 bits (taps as the reference makes them, in float32)."""
    w, d = np.float32(wavelength), np.float32(dT)
    pulse, cycle = int(np.float32(CYCLES) * w / d), int(w / d)
    sigma = np.float32(CYCLES) * w / np.float32(6)
    denom = float(np.float32(2) * sigma * sigma)
    k = np.arange(1, pulse + 1, dtype=np.float64)
    g = np.exp(-(float(d) * (k - pulse / 2.0)) ** 2 / denom)
    prog = 2.0 * math.pi * ((1.0 / cycle) * k)
    c = (np.cos(prog).astype(np.float32) * g).astype(np.float32)
    s = (np.sin(prog).astype(np.float32) * g).astype(np.float32)
    x = H.clone()
    x[:, 0] = 0.0                                       # bin 0 is never read
    x = torch.nn.functional.pad(x, (pulse // 2, pulse))
    out = torch.zeros(H.shape, dtype=torch.complex128, device="cuda")
    for j in range(pulse):
        out += x[:, j:j + H.shape[1]] * complex(float(c[j]), float(s[j]))
    return out


def _window(H, pairs, N, t0, dT):
    """The CPU path's volume: bins of the voxel-diagonal window around each path, in 64 bits."""
    dev, f = torch.device("cuda"), np.float32
    vs = VOLUME_SIZE / np.array(N, f)
    zero = VOLUME_POSITION - VOLUME_SIZE / f(2)
    half = f(np.sqrt(float(vs[0] * vs[0]) + float(vs[1] * vs[1]) + float(vs[2] * vs[2]))) / f(2)
    i = np.meshgrid(*[np.arange(n, dtype=f) for n in N], indexing="ij")
    v = torch.tensor(np.stack([zero[k] + i[k] * vs[k] for k in range(3)], -1).reshape(-1, 3).astype(np.float64), device=dev)
    lp, cp = (torch.tensor(pairs[k].astype(np.float64), device=dev) for k in ("laser_point", "camera_point"))
    lw, cw = (torch.tensor(pairs[k].astype(np.float64), device=dev) for k in ("laser_wall", "camera_wall"))
    T, t0, dT, half = H.shape[1], float(f(t0)), float(f(dT)), float(half)
    PS = torch.nn.functional.pad(H.cumsum(1), (1, 0))
    out = torch.zeros(len(v), dtype=torch.float64, device=dev)

    def dist(pts):
        d = [_f32(pts[:, None, k] - v[None, :, k]) for k in range(3)]
        return ((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]).sqrt()

    def edge(t):
        q = _f32(_f32(t - t0) / dT)
        return torch.where(q >= 0, torch.floor(q + 0.5), torch.ceil(q - 0.5)).clamp(0, T - 1).long()

    step = max(1, (1 << 25) // len(v))
    for p in range(0, len(lp), step):
        e = min(len(lp), p + step)
        total = _f32(_f32(lw[p:e, None] + _f32(dist(lp[p:e]) + dist(cp[p:e]))) + cw[p:e, None])
        a, b = edge(_f32(total - half)), edge(_f32(total + half))
        x = torch.gather(PS[p:e], 1, b) - torch.gather(PS[p:e], 1, a)
        out += torch.where(b > a, x, 0.0).sum(0)
    return out.reshape(tuple(N)).cpu()


def exact(case, seed):
    if case["kind"] == "octree":
        return None            # which voxels are reached follows from the proposal net's 16-bit layers
    if case["kind"] == "batch":
        out = []
        for i, m in enumerate(_batch_members(case, seed)):
            H, pairs, _, _ = _capture(m, 100 * seed + i)
            out.append(_single_tap(torch.as_tensor(H).double(), pairs, *_volume_grid(m), 0.0, RANGE / m["T"]))
        return out
    if _pairs_of(case) * case["nx"] * case["ny"] * case["nz"] > 6.0e10:
        return None            # minutes of work
    H, pairs, cg, lg = _capture(case, seed)
    N, zero, inc = _volume_grid(case)
    dT = RANGE / case["T"]
    if case["kind"] == "plan":
        return _single_tap(torch.as_tensor(H).double(), pairs, N, zero, inc, 0.0, dT)
    lo, hi = _time_limits(cg, lg, dT)
    if case["kind"] == "phasor":
        lo, hi = np.float32(int(lo)), np.float32(int(hi))
    chunk = _chunk(H, lo, hi)
    t0 = np.float32(0.0) + lo * np.float32(dT)
    if case["kind"] == "phasor":
        return _single_tap(_phasor_rows(chunk, case["wavelength"], dT), pairs, N, zero, inc, t0, dT)
    if case["kind"] == "window":
        return _window(chunk, pairs, N, t0, dT)
    return _single_tap(chunk, pairs, N, zero, inc, t0, dT)
