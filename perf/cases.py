"""Workloads of the library as its users run them: grids advanced by a frame
of CFL steps and batches of uneven patches, over the range of sizes, number
types and switches of the configurations, tests and benchmark.

Each case is one frame of a program that keeps its state in HBM: the state is
handed over as device buffers, advanced through ``advance`` (boundary pass,
CFL, step, per step) and taken back into device buffers.  A program of the
mixed form, whose fluxes are FP32, keeps its frames as FP32.  A batch is
advanced where it is and its patches are read back one by one.

``exact`` restates the schemes (MUSCL-Hancock, CTU, HLLC / HLLD, constrained
transport, Strang splitting) in plain FP64 torch, whole arrays at a time.
"""
import math
import random

import numpy as np
import torch

import dragon_amd as D

DEV = "cuda:0"
LIMITERS = {"minmod": 0, "mc": 1, "vanleer": 2, "superbee": 3, "vanalbada": 4}


def _case(name, problem, shape, steps, mhd, limiter, precision="fp64", gamma=5.0 / 3.0, bc="periodic", split=False, ct="beta"):
    n = list(shape) + [0, 0]
    return {"name": name, "problem": problem, "nx": n[0], "ny": n[1], "nz": n[2], "steps": steps, "mhd": mhd, "limiter": limiter,
            "precision": precision, "gamma": gamma, "bc": bc, "split": split, "ct": ct}


def _batch(name, patches, steps, precision, graph, lo=32, hi=256, bc="outflow"):
    return {"name": name, "problem": "batch", "patches": patches, "steps": steps, "precision": precision, "graph": graph, "lo": lo, "hi": hi,
            "bc": bc}


def listed():
    return [
        # the smallest calls: a shock tube of the 1D tests and examples, where launches and waits count
        _case("sod1d_1024", "sod", (1024,), 20, False, "minmod", bc="outflow"),
        # a 2D MHD grid of the size the tests and the child grids of a decomposition have
        _case("ot2d_128", "ot", (128, 128), 8, True, "mc"),
        # the small 3D MHD grid of the published accuracy table (field loop, n = 64), ct_energy off
        _case("loop3d_64", "loop", (64, 32, 32), 6, True, "mc", ct="total"),
        # 2D hydro at the benchmark configuration's size
        _case("kh2d_1024", "kh", (1024, 1024), 6, False, "vanleer"),
        # 2D hydro run with DIMENSION_UNSPLIT off, ragged sides
        _case("kh2d_split_1000x611", "kh", (1000, 611), 6, False, "mc", split=True),
        # 2D MHD, ragged sides, outflow: the rotor example on one grid
        _case("rotor2d_771x530", "rotor", (771, 530), 5, True, "minmod", gamma=1.4, bc="outflow"),
        # 2D MHD at the benchmark configuration's size, mixed form
        _case("ot2d_2048_mixed", "ot", (2048, 2048), 4, True, "mc", "mixed"),
        # 3D hydro (12-solve CTU), ragged sides
        _case("hydro3d_150x128x170", "turb", (150, 128, 170), 3, False, "vanleer"),
        # 3D MHD turbulence, the drop-in FP64 form, ragged sides
        _case("turb3d_240x200x261", "turb", (240, 200, 261), 2, True, "vanleer"),
        # the largest: the headline workload's mixed form, as large as three states fit
        _case("turb3d_384_mixed", "turb", (384, 384, 384), 2, True, "vanleer", "mixed"),
        # uneven 2D MHD patches, each with its own dt: FP64 launched eagerly, mixed replayed from a graph
        _batch("batch_96_fp64", 96, 80, "fp64", False),
        _batch("batch_192_mixed", 192, 100, "mixed", True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    lim = rng.choice(sorted(LIMITERS))
    prec = rng.choice(["fp64", "mixed"])
    kind = rng.choice(["sod", "hydro2d", "split2d", "mhd2d", "mhd2d", "hydro3d", "mhd3d", "mhd3d", "batch"])
    if kind == "sod":
        return _case("", "sod", (_log_int(rng, 200, 60000),), 20, False, lim, bc="outflow")
    if kind in ("hydro2d", "split2d"):
        n = _log_int(rng, 64, 1800)
        return _case("", "kh", (n, max(40, int(n * rng.uniform(0.5, 1.1)))), rng.randint(3, 6), False, lim, prec, split=kind == "split2d")
    if kind == "mhd2d":
        n = _log_int(rng, 64, 2048)
        m = max(40, int(n * rng.uniform(0.5, 1.0)))
        if rng.random() < 0.5:
            return _case("", "ot", (n, m), 4, True, lim, prec, ct=rng.choice(["beta", "total", "thermal"]))
        return _case("", "rotor", (n, m), 4, True, rng.choice(["minmod", "mc", "vanleer"]), prec, gamma=1.4, bc="outflow")
    if kind == "hydro3d":
        n = _log_int(rng, 32, 170)
        return _case("", "turb", (n, max(24, int(n * rng.uniform(0.6, 1.1))), max(24, int(n * rng.uniform(0.6, 1.1)))), 2, False, lim, prec)
    if kind == "mhd3d":
        n = _log_int(rng, 32, 280)
        m, k = (max(24, int(n * rng.uniform(0.6, 1.1))) for _ in range(2))
        return _case("", "turb", (n, m, k), 2, True, lim, prec, ct=rng.choice(["beta", "total"]))
    return _batch("", _log_int(rng, 24, 180), rng.randint(20, 40), prec, rng.random() < 0.5, hi=rng.randint(120, 256),
                  bc=rng.choice(["outflow", "periodic"]))


# ------------------------------------------------------------ initial states
def _shape(c):
    return tuple(c[k] for k in ("nx", "ny", "nz") if c[k])


def _spacing(c):
    shape = _shape(c)
    return (2.0 / shape[0],) * len(shape) if c["problem"] == "loop" else tuple(1.0 / n for n in shape)


def _ghosts(c):
    return 3 if c["mhd"] else 2


def initial_state(c, seed):
    """(W[8, ghosted shape], B[3, ghosted shape + 1] or None), interior set."""
    r = random.Random(seed)
    shape, d, g = _shape(c), _spacing(c), _ghosts(c)
    dim = len(shape)
    f64 = {"dtype": torch.float64, "device": DEV}
    W = torch.zeros((8,) + tuple(n + 2 * g for n in shape), **f64)
    wi = W[(slice(None),) + tuple(slice(g, g + n) for n in shape)]
    B = torch.zeros((3,) + tuple(n + 1 + 2 * g for n in shape), **f64) if c["mhd"] and dim >= 2 else None
    bi = None if B is None else B[(slice(None),) + tuple(slice(g, g + n + 1) for n in shape)]

    def along(v, ax):
        return v.reshape([-1 if q == ax else 1 for q in range(dim)])

    ctr = [along((torch.arange(n, **f64) + 0.5) * h, q) for q, (n, h) in enumerate(zip(shape, d))]
    two_pi = 2 * math.pi
    if c["problem"] == "sod":
        left = ctr[0] < r.uniform(0.4, 0.6)
        rho, p = r.uniform(0.1, 0.15), r.uniform(0.08, 0.15)
        wi[0] = torch.where(left, 1.0, rho)
        wi[1] = torch.where(left, 1.0, p)
    elif c["problem"] == "kh":
        gen = torch.Generator(device=DEV).manual_seed(seed)
        band = ((ctr[1] - 0.5).abs() < r.uniform(0.22, 0.28)).expand(shape)
        noise = (torch.rand((2,) + shape, generator=gen, **f64) * 2 - 1) * 0.01
        wi[0] = torch.where(band, 2.0, 1.0)
        wi[1] = 2.5
        wi[2] = torch.where(band, 0.5, -0.5) + noise[0]
        wi[3] = noise[1]
    elif c["problem"] == "ot":
        s, ph, qh = r.uniform(0.9, 1.1) / math.sqrt(4 * math.pi), r.uniform(0, two_pi), r.uniform(0, two_pi)
        wi[0] = 25.0 / (36.0 * math.pi)
        wi[1] = 5.0 / (12.0 * math.pi)
        wi[2] = -torch.sin(two_pi * ctr[1] + ph)
        wi[3] = torch.sin(two_pi * ctr[0] + qh)
        x, y = ((torch.arange(n + 1, **f64) + 0.5) / n for n in shape)
        bi[0] = (-torch.sin(two_pi * y + ph) * s)[None, :]
        bi[1] = (torch.sin(2 * two_pi * x + 2 * qh) * s)[:, None]
    elif c["problem"] == "rotor":
        b0, r0, u0 = r.uniform(2.5, 5.0), r.uniform(0.08, 0.12), r.uniform(1.0, 2.0)
        # off the middle: at a cell that rests, rounding alone would choose the upwind side of its EMF
        x, y = ctr[0] - r.uniform(0.47, 0.53), ctr[1] - r.uniform(0.47, 0.53)
        rad = torch.sqrt(x * x + y * y)
        r1 = 1.15 * r0
        f = ((r1 - rad) / (r1 - r0)).clamp(0.0, 1.0)
        inside = rad < r0
        wi[0] = torch.where(inside, 10.0, 1.0 + 9.0 * f)
        wi[1] = 1.0
        spin = torch.where(inside, u0 / r0, u0 * f / rad.clamp(min=1e-30))
        wi[2] = -spin * y
        wi[3] = spin * x
        bi[0] = b0 / math.sqrt(4 * math.pi)
    elif c["problem"] == "turb":
        modes = [k for k in ((a, b, e) for a in range(5) for b in range(-4, 5) for e in range(-4, 5)) if 1 <= sum(q * q for q in k) <= 16]
        for k in r.sample(modes, 12):
            kk = sum(q * q for q in k)
            amp = [r.gauss(0, 1) for _ in range(3)]
            dot = sum(a * q for a, q in zip(amp, k)) / kk
            amp = [(a - q * dot) / math.sqrt(kk) for a, q in zip(amp, k)]
            e = [torch.exp(2j * math.pi * q * x.to(torch.complex128)) for q, x in zip(k, ctr)]
            e[0] = e[0] * complex(math.cos(r.uniform(0, two_pi)), math.sin(r.uniform(0, two_pi)))
            a, b = e[0], e[1] * e[2]
            phase = a.real * b.real - a.imag * b.imag
            for q in range(3):
                wi[2 + q] += amp[q] * phase
            del phase
        wi[2:5] *= math.sqrt(c["gamma"]) / torch.sqrt(sum((v * v).mean() for v in wi[2:5])).item()
        wi[0] = 1.0
        wi[1] = 1.0
        if bi is not None:
            bi[0] = r.uniform(0.15, 0.25)
    elif c["problem"] == "loop":
        wi[0] = 1.0
        wi[1] = 5.0
        for q, v in enumerate((2.0, 1.0, 1.0)[:dim]):
            wi[2 + q] = v
        e = [along(torch.arange(n + 2, **f64) * h, q) for q, (n, h) in enumerate(zip(shape, d))][:2]
        rad = torch.sqrt((e[0] - 1.0) ** 2 + (e[1] - 0.5) ** 2)
        az = 1e-6 * (r.uniform(0.15, 0.25) - rad).clamp(min=0.0)  # B = curl(Az z)
        bi[0] = (az[:-1, 1:] - az[:-1, :-1]) / d[1]
        bi[1] = -(az[1:, :-1] - az[:-1, :-1]) / d[0]
    else:
        raise ValueError(c["problem"])
    return W, B


def _batch_patches(c, seed):
    """Per patch: side, and the rotor's (B0, r0, u0) and centre."""
    r = random.Random(seed)
    sizes = random.Random(1234567)  # the decomposition is the program's, the states are the seed's
    out = []
    for _ in range(c["patches"]):
        nx = int(math.exp(sizes.uniform(math.log(c["lo"]), math.log(c["hi"]))))
        ny = max(16, min(c["hi"] - 1, int(nx * sizes.uniform(0.8, 1.25))))
        out.append((nx, ny, r.uniform(2.5, 5.0), r.uniform(0.08, 0.12), r.uniform(1.0, 2.0), r.uniform(0.47, 0.53), r.uniform(0.47, 0.53)))
    return out


def _rotor_patch(nx, ny, b0, r0, u0, cx, cy, g=3):
    w, B = np.zeros((nx + 2 * g, ny + 2 * g, 8)), np.zeros((nx + 1 + 2 * g, ny + 1 + 2 * g, 3))
    x, y = ((np.arange(nx) + 0.5) / nx - cx)[:, None], ((np.arange(ny) + 0.5) / ny - cy)[None, :]
    rad = np.sqrt(x * x + y * y)
    f = np.clip((1.15 * r0 - rad) / (0.15 * r0), 0.0, 1.0)
    inside = rad < r0
    wi = w[g:-g, g:-g]
    wi[..., 0] = np.where(inside, 10.0, 1.0 + 9.0 * f)
    wi[..., 1] = 1.0
    spin = np.where(inside, u0 / r0, u0 * f / np.maximum(rad, 1e-30))
    wi[..., 2] = -spin * y
    wi[..., 3] = spin * x
    B[g:-g, g:-g, 0] = b0 / math.sqrt(4 * math.pi)
    return w, B


# ------------------------------------------------------------- the workloads
def _config(c):
    cfg = D.Config(mhd=int(c.get("mhd", True)), gamma=c.get("gamma", 1.4), limiter=LIMITERS[c.get("limiter", "minmod")],
                   precision=D.MIXED if c["precision"] == "mixed" else D.FP64, dimension_unsplit=int(not c.get("split", False)))
    cfg.ct_energy = {"beta": D.CT_CONSV_BETA_GATED, "total": D.CT_CONSV_TOTAL_E, "thermal": D.CT_CONSV_THERMAL}[c.get("ct", "beta")]
    return cfg


def prepare(case, seed):
    cfg = _config(case)
    if case["problem"] == "batch":
        patches = _batch_patches(case, seed)
        b = D.Batch([p[:2] for p in patches], [(1.0 / p[0], 1.0 / p[1]) for p in patches], cfg, bc=case["bc"])
        for q, p in enumerate(patches):
            b.set_state(q, *_rotor_patch(*p))
        b.initialize_B_fields()
        return {"case": case, "batch": b}
    shape, d = _shape(case), _spacing(case)
    G = D.Grid(shape, d, 1, cfg)
    if case["bc"] == "periodic":
        G.boundary = D.Periodic()
    W, B = initial_state(case, seed)
    torch.cuda.synchronize()
    if B is not None:  # cell-centred B of the faces, once
        G.upload_device(W.data_ptr(), B.data_ptr())
        G.initialize_B_fields()
        G.download_device(W.data_ptr(), B.data_ptr())
    s = {"case": case, "grid": G, "W": W, "B": B, "Wo": torch.empty_like(W), "Bo": None if B is None else torch.empty_like(B)}
    if case["precision"] == "mixed":
        s["W32"] = torch.empty_like(W, dtype=torch.float32)
        s["B32"] = None if B is None else torch.empty_like(B, dtype=torch.float32)
        s["stream"] = torch.cuda.ExternalStream(G.stream, device=DEV)
    return s


def run(state):
    c = state["case"]
    if c["problem"] == "batch":
        b = state["batch"]
        b.run(c["steps"], graph=c["graph"])
        b.sync()
        got = [b.get_state(p) for p in range(b.n)]
        kind = np.float32 if c["precision"] == "mixed" else np.float64
        return {"cells": np.concatenate([w.reshape(-1) for w, _ in got], dtype=kind, casting="same_kind"),
                "faces": np.concatenate([B.reshape(-1) for _, B in got], dtype=kind, casting="same_kind")}
    G, W, B, Wo, Bo = state["grid"], state["W"], state["B"], state["Wo"], state["Bo"]
    G.upload_device(W.data_ptr(), None if B is None else B.data_ptr())
    G.advance(1e9, True, c["steps"])
    G.download_device(Wo.data_ptr(), None if B is None else Bo.data_ptr())
    if c["precision"] == "mixed":
        with torch.cuda.stream(state["stream"]):
            Wo = state["W32"].copy_(Wo)
            Bo = None if B is None else state["B32"].copy_(Bo)
    return {"cells": Wo} if B is None else {"cells": Wo, "faces": Bo}


def work(case):
    """Per step the state read once and written once (5 fields of a hydro
    cell, 8 of an MHD one, faces among them, FP64) and about this many
    additions, products, divisions and square roots a zone: one
    reconstruction and two Riemann solves per axis (three and a third in 3D
    hydro's CTU), the CTU and constrained-transport terms, the update."""
    if case["problem"] == "batch":
        zones = sum(p[0] * p[1] for p in _batch_patches(case, 0))
        return {"bytes": 128 * zones * case["steps"], "flops": 2400 * zones * case["steps"]}
    shape = _shape(case)
    zones, dim = math.prod(shape) * case["steps"], len(shape)
    if case["mhd"]:
        return {"bytes": 128 * zones, "flops": {2: 2400, 3: 3900}[dim] * zones}
    if case["split"]:
        return {"bytes": 80 * zones, "flops": 250 * (2 * dim - 1) * zones}
    return {"bytes": 80 * zones, "flops": {1: 250, 2: 800, 3: 2600}[dim] * zones}


# ------------------------------------------------- the schemes in plain FP64
# A record is a list of fields: primitive [rho, p, vx, vy, vz, Bx, By, Bz],
# conserved / flux [rho, E, mx, my, mz, Bx, By, Bz]; hydro has the first five.
# Directional work is done with the axis' components first (_turn).
K4, K8 = 0.25 / math.pi, 0.125 / math.pi
SQ4PI = math.sqrt(4 * math.pi)


def _sh(a, ax, k):
    """b[i] = a[i + k] along ax."""
    return torch.roll(a, -k, ax)


def _turn(w, ax):
    o = {0: (0, 1, 2), 1: (1, 0, 2), 2: (2, 1, 0)}[ax]
    return w[:2] + [w[2 + q] for q in o] + [w[5 + q] for q in o if len(w) > 5]


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _cons(w, gam):
    E = w[1] / (gam - 1) + 0.5 * w[0] * _dot(w[2:5], w[2:5])
    if len(w) > 5:
        E = E + _dot(w[5:], w[5:]) * K8
    return [w[0], E] + [w[0] * v for v in w[2:5]] + list(w[5:])


def _prim(u, gam):
    e = u[1] - _dot(u[2:5], u[2:5]) / (2 * u[0])
    if len(u) > 5:
        e = e - _dot(u[5:], u[5:]) * K8
    return [u[0], (gam - 1) * e] + [m / u[0] for m in u[2:5]] + list(u[5:])


def _flux(w, u):
    """Physical flux along the first component."""
    vx, p = w[2], w[1]
    F = [u[2], (u[1] + p) * vx, u[2] * vx + p, u[3] * vx, u[4] * vx]
    if len(w) > 5:
        pm = _dot(w[5:], w[5:]) * K8
        t = [b * w[5] * K4 for b in w[5:]]
        F[1] = F[1] + pm * vx - _dot(w[2:5], t)
        F[2] = F[2] + pm - t[0]
        F[3] = F[3] - t[1]
        F[4] = F[4] - t[2]
        F += [torch.zeros_like(vx), w[6] * vx - w[3] * w[5], w[7] * vx - w[4] * w[5]]
    return F


def _physical(w):
    ok = (w[0] > 0) & (w[1] > 0)
    for f in w:
        ok = ok & torch.isfinite(f)
    return ok


def _minmod(a, b):
    return torch.where(a * b <= 0, 0.0, torch.where(a.abs() < b.abs(), a, b))


def _limit(a, b, lim):
    if lim == "minmod":
        return _minmod(a, b)
    if lim == "mc":
        c = (a + b).abs()
        s = torch.where((c < 4 * a.abs()) & (c < 4 * b.abs()), 0.5 * (a + b), 2 * _minmod(a, b))
    elif lim == "vanleer":
        s = 2 * a * b / (a + b)
    elif lim == "superbee":
        A, C = a.abs(), b.abs()
        s = torch.maximum(torch.minimum(2 * A, C), torch.minimum(A, 2 * C)) * torch.sign(a)
    else:
        s = a * b * (a + b) / (a * a + b * b)
    return torch.where(a * b <= 0, 0.0, s)


def _muscl(wl, wc, wr, dt_d, dB, gam, lim):
    """Half states (low side, high side) of the cells, MUSCL-Hancock."""
    s = [_limit(c - a, b - c, lim) for a, c, b in zip(wl, wc, wr)]
    lo, hi = [c - 0.5 * q for c, q in zip(wc, s)], [c + 0.5 * q for c, q in zip(wc, s)]
    ul, uh = _cons(lo, gam), _cons(hi, gam)
    corr = [0.5 * dt_d * (b - a) for a, b in zip(_flux(lo, ul), _flux(hi, uh))]
    if len(wc) > 5:
        a_s = (hi[5] - lo[5]) * dt_d
        dy = 0.5 * wc[3] * _minmod(dB[0], -dB[1]) - 0.25 * (lo[3] + hi[3]) * a_s
        dz = 0.5 * wc[4] * _minmod(dB[0], -dB[2]) - 0.25 * (lo[4] + hi[4]) * a_s
        corr[6] = corr[6] - dy
        corr[7] = corr[7] - dz
        corr[1] = corr[1] - K4 * (wc[6] * dy + wc[7] * dz)
    lo, hi = _prim([u - q for u, q in zip(ul, corr)], gam), _prim([u - q for u, q in zip(uh, corr)], gam)
    ok = _physical(lo) & _physical(hi)
    return [torch.where(ok, a, c) for a, c in zip(lo, wc)], [torch.where(ok, a, c) for a, c in zip(hi, wc)]


def _sel(c, a, b):
    return [torch.where(c, x, y) for x, y in zip(a, b)]


def _fast(w, gam):
    c2, a2, ax2 = gam * w[1] / w[0], _dot(w[5:], w[5:]) / w[0] * K4, w[5] * w[5] / w[0] * K4
    return torch.sqrt(0.5 * (c2 + a2) + torch.sqrt((0.25 * (c2 + a2) ** 2 - ax2 * c2).clamp(min=0.0)))


def _hll(L, R, sl, sr, gam):
    UL, UR = _cons(L, gam), _cons(R, gam)
    FL, FR = _flux(L, UL), _flux(R, UR)
    M = [(fl * sr - fr * sl + (ur - ul) * (sl * sr)) / (sr - sl) for fl, fr, ul, ur in zip(FL, FR, UL, UR)]
    return _sel(sl >= 0, FL, _sel(sr <= 0, FR, M))


def _hlle(L, R, gam):
    ql, qr = torch.sqrt(L[0]), torch.sqrt(R[0])
    a, b = ql / (ql + qr), qr / (ql + qr)
    al, ar = _fast(L, gam), _fast(R, gam)
    d = torch.sqrt(a * al * al + b * ar * ar + 0.5 * ql * qr * ((R[2] - L[2]) / (ql + qr)) ** 2)
    u = a * L[2] + b * R[2]
    return _hll(L, R, torch.minimum(L[2] - al, u - d), torch.maximum(R[2] + ar, u + d), gam)


def _hllc(L, R, gam):
    ql, qr = torch.sqrt(L[0]), torch.sqrt(R[0])
    a, b = ql / (ql + qr), qr / (ql + qr)
    UL, UR = _cons(L, gam), _cons(R, gam)
    v = [a * x + b * y for x, y in zip(L[2:5], R[2:5])]
    H = a * (UL[1] + L[1]) / L[0] + b * (UR[1] + R[1]) / R[0]
    am = torch.sqrt((gam - 1) * (H - 0.5 * _dot(v, v)))
    sl = torch.minimum(L[2] - torch.sqrt(gam * L[1] / L[0]), v[0] - am)
    sr = torch.maximum(R[2] + torch.sqrt(gam * R[1] / R[0]), v[0] + am)
    pr, pl = R[1] + R[0] * R[2] * (R[2] - sr), L[1] + L[0] * L[2] * (L[2] - sl)
    sc = (pr - pl) / (R[0] * (R[2] - sr) - L[0] * (L[2] - sl))
    left = sc > 0
    X, U, sx = _sel(left, L, R), _sel(left, UL, UR), torch.where(left, sl, sr)
    S = [q * (sx - X[2]) / (sx - sc) for q in U]
    S[2] = S[0] * sc
    S[1] = S[1] + S[0] * (sc - X[2]) * (sc + X[1] / (X[0] * (sx - X[2])))
    M = [f + sx * (s - u) for f, s, u in zip(_flux(X, U), S, U)]
    return _sel(sl >= 0, _flux(L, UL), _sel(sr <= 0, _flux(R, UR), M))


def _hlld(L, R, gam):
    Bx = 0.5 * (L[5] + R[5])
    L, R = L[:5] + [Bx] + L[6:], R[:5] + [Bx] + R[6:]
    cl, cr = _fast(L, gam), _fast(R, gam)
    SL, SR = torch.minimum(L[2] - cl, R[2] - cr), torch.maximum(L[2] + cl, R[2] + cr)
    bl, br = _dot(L[5:], L[5:]), _dot(R[5:], R[5:])
    zero = Bx * Bx < 1e-12 * (bl + br).clamp(min=1e-100)
    ptl, ptr = L[1] + bl * K8, R[1] + br * K8
    xl, xr = L[0] * (SL - L[2]), R[0] * (SR - R[2])
    SM = ((xr * R[2] - xl * L[2]) - (ptr - ptl)) / (xr - xl)
    pT = (xr * ptl - xl * ptr + xl * xr * (R[2] - L[2])) / (xr - xl)
    UL, UR = _cons(L, gam), _cons(R, gam)

    def star(K, U, x, S, pt):
        rho = x / (S - SM)
        bx2 = Bx * Bx * K4
        den = x * (S - SM) - bx2
        tiny = den.abs() < 1e-12
        s = (x * (S - K[2]) - bx2) / den
        t = (SM - K[2]) / den * Bx * K4
        B = [Bx] + [torch.where(tiny, b, b * s) for b in K[6:]]
        v = [SM] + [torch.where(tiny, w, w - b * t) for w, b in zip(K[3:5], K[6:])]
        zt = (S - SM).abs() < 1e-12
        B0 = [torch.zeros_like(Bx)] + [torch.where(zt, b, b * (S - K[2]) / (S - SM)) for b in K[6:]]
        B, v = _sel(zero, B0, B), _sel(zero, [SM] + K[3:5], v)
        E = U[1] * (S - K[2]) + pT * SM - pt * K[2]
        E = E + torch.where(zero, 0.0, Bx * (_dot(K[2:5], K[5:]) - _dot(v, B)) * K4)
        E = E / (S - SM)
        w = [rho, pT - _dot(B, B) * K8] + v + B
        return w, [rho, E] + [rho * q for q in v] + B

    wl, ul = star(L, UL, xl, SL, ptl)
    wr, ur = star(R, UR, xr, SR, ptr)

    def good(w, u):
        ok = _physical(w) & (zero | (_prim(u, gam)[1] > 0))
        for q in u:
            ok = ok & torch.isfinite(q)
        return ok

    okl, okr = good(wl, ul), good(wr, ur)
    ssl = SM - Bx.abs() / (SQ4PI * torch.sqrt(ul[0]))
    ssr = SM + Bx.abs() / (SQ4PI * torch.sqrt(ur[0]))
    ql, qr = torch.sqrt(wl[0]), torch.sqrt(wr[0])
    a, b = ql / (ql + qr), qr / (ql + qr)
    FL, FR = _flux(L, UL), _flux(R, UR)
    fl, fr = [f + SL * (s - u) for f, s, u in zip(FL, ul, UL)], [f + SR * (s - u) for f, s, u in zip(FR, ur, UR)]
    fl[5], fr[5] = torch.zeros_like(Bx), torch.zeros_like(Bx)
    # double star
    right = SM >= 0
    ws, us = _sel(right, wl, wr), _sel(right, ul, ur)
    sg = torch.sign(Bx) * SQ4PI
    vy, vz = (wl[q] * a + wr[q] * b + (ur[q + 3] - ul[q + 3]) * sg * K4 / (ql + qr) for q in (3, 4))
    by, bz = (ur[q + 3] * a + ul[q + 3] * b + (wr[q] - wl[q]) * sg * ql * qr / (ql + qr) for q in (3, 4))
    v2, b2 = [SM, vy, vz], [Bx, by, bz]
    dE = sg * (_dot(ws[2:5], ws[5:]) - _dot(v2, b2)) * K4 * torch.sqrt(ws[0])
    u2 = [ws[0], torch.where(right, ul[1] - dE, ur[1] + dE)] + [ws[0] * q for q in v2] + b2
    f2 = [f + torch.where(right, ssl, ssr) * (p - q) for f, p, q in zip(_sel(right, fl, fr), u2, us)]
    ok2 = _physical([ws[0], pT - _dot(b2, b2) * K8] + v2 + b2) & torch.isfinite(u2[1])
    inner = ~(ssl >= 0) & ~(ssr <= 0)
    ok = (okl | ~(ssr >= 0)) & (okr | ~(ssl <= 0)) & (ok2 | ~inner)
    F = _sel(ssl >= 0, fl, _sel(ssr <= 0, fr, f2))
    mean = [a * p + b * q for p, q in zip(fl, fr)]
    F = _sel(zero, _sel(SM > 0, fl, _sel(SM < 0, fr, mean)), F)
    ok = torch.where(zero, (okl | (SM < 0)) & (okr | (SM > 0)), ok)
    if not bool(ok.all()):
        F = _sel(ok, F, _hlle(L, R, gam))
    return _sel(SL >= 0, FL, _sel(SR <= 0, FR, F))


class _Exact:
    """One grid.  Every array has the face arrays' shape (one more than the
    ghosted cells); whole arrays are computed and the wrapped margins, which
    no interior cell depends on, are dropped at the commit."""

    def __init__(self, c, W, B):
        self.c, self.gam, self.lim = c, c["gamma"], c["limiter"]
        self.shape, self.d, self.g = _shape(c), _spacing(c), _ghosts(c)
        self.dim, self.mhd = len(self.shape), B is not None
        pad = [0, 1] * self.dim
        self.nf = 8 if self.mhd else 5
        self.w = [torch.nn.functional.pad(f[None, None], pad, mode="replicate")[0, 0] for f in W[: self.nf]]
        self.B = None if B is None else [f.clone() for f in B]
        self.turn = 0

    def cells(self):
        return [f[(slice(None, -1),) * self.dim] for f in self.w]

    # boundary: one axis after the other, over everything the other axes hold
    def fill(self):
        g = self.g
        at = lambda f, ax, i: f.narrow(ax, g + i, 1)  # noqa: E731
        for ax in range(self.dim):
            n = self.shape[ax]
            for f in self.w:
                for q in range(1, g + 1):
                    lo, hi = (n - q, q - 1) if self.c["bc"] == "periodic" else (0, n - 1)
                    at(f, ax, -q).copy_(at(f, ax, lo))
                    at(f, ax, n - 1 + q).copy_(at(f, ax, hi))
        for ax in range(self.dim if self.mhd else 0):
            n = self.shape[ax]
            for q, f in enumerate(self.B):
                if self.c["bc"] == "periodic":
                    for k in range(1, g + 1):
                        at(f, ax, -k).copy_(at(f, ax, n - k))
                        at(f, ax, n - 1 + k).copy_(at(f, ax, k - 1))
                    continue
                if q != ax:
                    at(f, ax, n).copy_(at(f, ax, n - 1))
                for k in range(1, g + 1):
                    if q == ax:
                        at(f, ax, -k).copy_(2 * at(f, ax, -k + 1) - at(f, ax, -k + 2))
                        at(f, ax, n + k).copy_(2 * at(f, ax, n + k - 1) - at(f, ax, n + k - 2))
                    else:
                        at(f, ax, -k).copy_(at(f, ax, 0))
                        at(f, ax, n + k).copy_(at(f, ax, n))

    def dt(self):
        g = self.g
        box = tuple(slice(g - 1, g + n + 1) for n in self.shape)
        w = [f[box] for f in self.w]
        if self.mhd:
            b2 = [b * b for b in w[5:]]
            least = torch.minimum(torch.minimum(b2[0], b2[1]), b2[2])
            c2, a2 = self.gam * w[1] / w[0], (b2[0] + b2[1] + b2[2]) / w[0] * K4
            a = torch.sqrt(0.5 * (c2 + a2) + torch.sqrt((0.25 * (c2 + a2) ** 2 - least / w[0] * K4 * c2).clamp(min=0.0)))
        else:
            a = torch.sqrt(self.gam * w[1] / w[0])
        return 0.3 / sum((w[2 + q].abs() + a) / self.d[q] for q in range(self.dim)).max().item()

    def in_parts(self, fn, args, out):
        """fn over flattened pieces of the records `args`, `out` records of results."""
        like = args[0][0]
        res = [[torch.empty_like(like) for _ in range(self.nf)] for _ in range(out)]
        step = 1 << 23
        for s in range(0, like.numel(), step):
            part = [[f.reshape(-1)[s:s + step] for f in r] for r in args]
            got = fn(*part)
            for r, q in zip(res, got if out > 1 else (got,)):
                for f, v in zip(r, q):
                    f.view(-1)[s:s + step] = v
        return res if out > 1 else res[0]

    def half_states(self, ax, dt_d, dB):
        w = _turn(self.w, ax)
        args = [[_sh(f, ax, -1) for f in w], w, [_sh(f, ax, 1) for f in w]]
        if self.mhd:
            args.append([dB[q] for q in {0: (0, 1, 2), 1: (1, 0, 2), 2: (2, 1, 0)}[ax]])
        lo, hi = self.in_parts(lambda a, b, c, e=None: _muscl(a, b, c, dt_d, e, self.gam, self.lim), args, 2)
        del args
        lo, hi = _turn(lo, ax), _turn(hi, ax)
        if self.mhd:
            lo[5 + ax], hi[5 + ax] = self.B[ax], _sh(self.B[ax], ax, 1)
        return lo, hi

    def solve(self, ax, lo, hi):
        solver = _hlld if self.mhd else _hllc
        L, R = _turn([_sh(f, ax, -1) for f in hi], ax), _turn(lo, ax)
        return _turn(self.in_parts(lambda a, b: solver(a, b, self.gam), [L, R], 1), ax)

    def emf(self, F, ref):
        """Corner EMF, Gardiner-Stone upwinding with the reference EMF `ref`."""

        def up(m, fm, fp, rm, rp):
            return torch.where(m > 1e-18, 0.25 * (fm - rm), torch.where(m < -1e-18, 0.25 * (fp - rp), 0.125 * (fm + fp - rm - rp)))

        if self.dim == 2:
            X, Y = F
            ex = -Y[7] + 0.25 * (-2 * Y[7] - ref[0] - _sh(ref[0], 1, -1))
            ey = X[7] + 0.25 * (2 * X[7] - ref[1] - _sh(ref[1], 0, -1))
            pairs = [(2, 0, 1)]
        else:
            ex = ey = None
            pairs = [(0, 1, 2), (1, 2, 0), (2, 0, 1)]
        E = [ex, ey, None]
        for e, a, b in pairs:  # E_e between the faces of a and b: +F_b[B_a], -F_a[B_b]
            fa, fb, r = F[a], F[b], ref[e]
            pa, pb = fb[5 + a], -fa[5 + b]
            pal, pbl, rl = _sh(pa, a, -1), _sh(pb, b, -1), _sh(r, a, -1)
            v = 0.25 * (pal + pa + pbl + pb)
            v = v + up(fa[0], pal, pa, rl, r)
            v = v + up(_sh(fa[0], b, -1), pal, pa, _sh(rl, b, -1), _sh(r, b, -1))
            v = v + up(fb[0], pbl, pb, _sh(r, b, -1), r)
            v = v + up(_sh(fb[0], a, -1), pbl, pb, _sh(rl, b, -1), rl)
            E[e] = v
        return E

    def curl(self, E, k):
        """dt curl E at the faces, k[q] = dt / d[q]."""
        diff = lambda q, ax: (_sh(E[q], ax, 1) - E[q]) * k[ax]  # noqa: E731
        if self.dim == 2:
            return [diff(2, 1), -diff(2, 0), diff(1, 0) - diff(0, 1)]
        return [diff(2, 1) - diff(1, 2), diff(0, 2) - diff(2, 0), diff(1, 0) - diff(0, 1)]

    def centre(self, B):
        return [0.5 * (B[q] + _sh(B[q], q, 1)) if q < self.dim else B[q] for q in range(3)]

    def update(self, F, k, B):
        """Primitive state after the flux differences, cell B of the faces B."""
        u = _cons(self.w, self.gam)
        for ax in range(self.dim):
            for q in range(self.nf):
                if q != 5 + ax:
                    u[q] = u[q] + (F[ax][q] - _sh(F[ax][q], ax, 1)) * k[ax]
        w = _prim(u, self.gam)
        if B is None:
            return w
        cb = self.centre(B)
        total = _prim(u[:1] + [_cons(w, self.gam)[1]] + u[2:5] + cb, self.gam)
        if self.c["ct"] == "total":
            return total
        keep = w[:5] + cb
        if self.c["ct"] == "thermal":
            return keep
        b2 = _dot(w[5:], w[5:])
        return _sel((b2 != 0) & (8 * math.pi * w[1] / b2 <= 0.1), keep, total)

    def commit(self, w, curl=None):
        box = tuple(slice(self.g, self.g + n) for n in self.shape)
        for f, v in zip(self.w, w):
            f[box] = v[box]
        if curl is not None:
            for q in range(3):
                fb = tuple(slice(self.g, self.g + n + (1 if q == ax else 0)) for ax, n in enumerate(self.shape))
                self.B[q][fb] -= curl[q][fb]

    def unsplit(self, dt):
        k = [dt / h for h in self.d]
        D_ = range(self.dim)
        h = [0.5 * v for v in k]
        if not self.mhd:
            S = [self.half_states(ax, k[ax], None) for ax in D_]
            F = [self.solve(ax, *S[ax]) for ax in D_]

            def moved(ax, by, flux, dd):
                t = [(_sh(f, by, 1) - f) * dd for f in flux]
                return tuple(_prim([u - q for u, q in zip(_cons(s, self.gam), t)], self.gam) for s in S[ax])

            if self.dim == 2:
                S = [moved(0, 1, F[1], h[1]), moved(1, 0, F[0], h[0])]
            else:
                T = {(a, b): self.solve(a, *moved(a, b, F[b], k[b] / 3)) for a in D_ for b in D_ if a != b}
                del F
                for ax in D_:
                    a, b = [q for q in D_ if q != ax]
                    S[ax] = moved(ax, a, T[a, b], h[a])
                    S[ax] = moved(ax, b, T[b, a], h[b])
            F = [self.solve(ax, *S[ax]) for ax in D_]
            self.commit(self.update(F, k, None))
            return
        dB = [(_sh(self.B[q], q, 1) - self.B[q]) * k[q] if q < self.dim else torch.zeros_like(self.B[0]) for q in range(3)]
        S = [self.half_states(ax, k[ax], dB) for ax in D_]
        F = [self.solve(ax, *S[ax]) for ax in D_]
        w = self.w
        E = self.emf(F, torch.linalg.cross(torch.stack(w[5:]), torch.stack(w[2:5]), dim=0))
        Bh = [a - b for a, b in zip(self.B, self.curl(E, h))]
        m = self.update(F, h, Bh)
        ref = torch.linalg.cross(torch.stack(m[5:]), torch.stack(m[2:5]), dim=0)
        del m
        for ax in D_:
            c = [torch.zeros_like(w[0]) for _ in range(8)]
            for b in D_:
                if b != ax:
                    for q in range(5):
                        c[q] += h[b] * (F[b][q] - _sh(F[b][q], b, 1))
            for b in range(3):  # source terms and the EMF difference of each transverse component
                if b == ax:
                    continue
                other = 3 - ax - b
                if self.dim == 2 and b < 2:
                    continue  # the in-plane transverse field has none
                lim = _minmod(-dB[other], dB[ax])
                c[1] += K8 * w[5 + b] * w[2 + b] * lim
                sign = 1.0 if (b - ax) % 3 == 2 else -1.0
                if self.dim == 2:
                    e = 0.5 * sign * k[other] * (_sh(E[ax], other, 1) - E[ax])
                else:
                    dE = _sh(E[ax], other, 1) - E[ax]
                    e = 0.25 * sign * k[other] * (dE + _sh(dE, b, 1))
                c[5 + b] += e + 0.5 * w[2 + b] * lim
            lo, hi = ([u + q for u, q in zip(_cons(s, self.gam), c)] for s in S[ax])
            lo[5 + ax], hi[5 + ax] = Bh[ax], _sh(Bh[ax], ax, 1)
            S[ax] = (_prim(lo, self.gam), _prim(hi, self.gam))
        del F, Bh, dB
        F = [self.solve(ax, *S[ax]) for ax in D_]
        del S
        self.commit([], self.curl(self.emf(F, ref), k))  # the faces first: the update centres them
        self.commit(self.update(F, k, self.B))

    def sweep(self, ax, dt):
        """Godunov sweep of every line of an axis, ghost lines included: first
        order on the outermost cells, cells [-g+1, n+g-2] updated."""
        k, n, g = dt / self.d[ax], self.shape[ax], self.g
        lo, hi = self.half_states(ax, k, None)
        for i in (0, n + 2 * g - 1):
            for s in (lo, hi):
                for f, c in zip(s, self.w):
                    f.narrow(ax, i, 1).copy_(c.narrow(ax, i, 1))
        F = self.solve(ax, lo, hi)
        u = [a + (f - _sh(f, ax, 1)) * k for a, f in zip(_cons(self.w, self.gam), F)]
        for f, v in zip(self.w, _prim(u, self.gam)):
            f.narrow(ax, 1, n + 2 * g - 2).copy_(v.narrow(ax, 1, n + 2 * g - 2))

    def step(self):
        self.fill()
        dt = self.dt()
        if self.dim == 1:
            self.sweep(0, dt)
        elif self.c["split"]:
            a = self.turn % 2
            for q, (ax, t) in enumerate(((a, dt / 2), (1 - a, dt), (a, dt / 2))):
                if q:
                    self.fill()
                self.sweep(ax, t)
        else:
            self.unsplit(dt)
        self.turn += 1


def exact(case, seed):
    if case["problem"] == "batch":
        return None  # hundreds of grids, tens of steps each: minutes
    W, B = initial_state(case, seed)
    if case["mhd"] and B is not None:
        E = _Exact(case, W, B)
        E.fill()
        cb = E.centre(E.B)
        for q in range(3):
            E.w[5 + q] = cb[q]
    else:
        E = _Exact(case, W, B)
    for _ in range(case["steps"]):
        E.step()
    kind = torch.float64
    cells = torch.zeros_like(W, dtype=kind)
    for f, v in zip(cells, E.cells()):
        f.copy_(v)
    return {"cells": cells} if B is None else {"cells": cells, "faces": torch.stack(E.B)}
