"""The calls whose time this framework is judged by, from its public entry points.

A case is a dict of plain values; `kind` names the path:

  recover3d  CuWaveletPotentialRecover3D.Solve: a vector potential from a MAC velocity
             (3-array or, with `vout`, 6-array form)
  recover2d  CuWaveletPotentialRecover2D.Solve: the stream function of a 2D velocity
  batch      CuBatchRecover3D.Replay: many uneven grids in one captured graph
  solids     divergence, pressure solve and velocity correction around solid spheres
             (CuConvergence, CuMultigridFrac3D, CuGradient)
  geometry   level set, eikonal relaxations and face fractions
             (CuSolidLevelSet3D, CuFastSweeping)
  sweep      CuParallelSweep3D.Solve + Project: the sweep + DST comparator
  predict    UNet3D.predict: the learned initial guess
  train      UNet3D.loss_grad + adam + gradients read back: one training step

Inputs are made on the GPU in FP64 from the seed alone and rounded to the type
the path takes.  `exact` restates a path in FP64 with torch only, where the
result has a closed form or a short definition; a 3D potential has none (its
gauge is fixed by the wavelet projection), so only the returned velocity of the
`vout` form is given there.
"""
import math
import os
import random

import numpy as np
import torch

import waveletpotentials_amd as W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "waveletpotentials_amd", "weights", "unet_solids192.bin")
BATCH_GRIDS = ((32, 32, 32), (64, 64, 64), (128, 128, 128), (128, 64, 64))
PAIRS = {"cdf3.7": ("WT_CDF3_7", "WT_CDF4_6"), "cdf3.5": ("WT_CDF3_5", "WT_CDF4_4")}
F64 = torch.float64


def listed():
    return [
        # one small 2D flow per call: launch latency
        {"name": "recover2d 128^2", "kind": "recover2d", "nx": 128, "ny": 128},
        # a small 3D grid, as a test scene or a coarse level of an interactive tool
        {"name": "recover3d 32^3", "kind": "recover3d", "nx": 32, "ny": 32, "nz": 32, "bc": "n",
         "wavelet": "cdf3.7", "vout": False},
        # a channel with wall flux, the shorter wavelet pair, the projected velocity returned too
        {"name": "recover3d 128x64x32 d", "kind": "recover3d", "nx": 128, "ny": 64, "nz": 32,
         "bc": "d", "wavelet": "cdf3.5", "vout": True},
        # the production grid of the recovery
        {"name": "recover3d 256^3", "kind": "recover3d", "nx": 256, "ny": 256, "nz": 256,
         "bc": "n", "wavelet": "cdf3.7", "vout": False},
        # many simulations' grids at once, one graph per step
        {"name": "batch 64", "kind": "batch", "count": 64, "mix": 4},
        # pressure projection of a flow around solids, production size
        {"name": "solids 192^3 pcg", "kind": "solids", "nx": 192, "ny": 192, "nz": 192,
         "spheres": 8, "bc": "n", "method": "pcg"},
        # the same by V-cycles on a ragged box with open walls
        {"name": "solids 100x76x52 vcycles d", "kind": "solids", "nx": 100, "ny": 76, "nz": 52,
         "spheres": 3, "bc": "d", "method": "vcycles"},
        # the scene's solid geometry, once per moved solid
        {"name": "geometry 160x120x136", "kind": "geometry", "nx": 160, "ny": 120, "nz": 136,
         "spheres": 8},
        # the comparator at the production size (transform lengths of 2^8)
        {"name": "sweep 256^3", "kind": "sweep", "nx": 256, "ny": 256, "nz": 256, "bc": "n",
         "dtype": "f32"},
        # the comparator in FP64 on a ragged box (transform lengths with other factors)
        {"name": "sweep 96x80x60 d f64", "kind": "sweep", "nx": 96, "ny": 80, "nz": 60,
         "bc": "d", "dtype": "f64"},
        # the learned start of a 192^3 solve, network on 48^3
        {"name": "predict 192^3 f4", "kind": "predict", "nx": 192, "ny": 192, "nz": 192,
         "factor": 4},
        # one training step of that network
        {"name": "train 192^3 f4", "kind": "train", "nx": 192, "ny": 192, "nz": 192, "factor": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("recover3d", "recover3d", "recover3d", "recover2d", "batch", "solids",
                       "solids", "geometry", "sweep", "sweep", "predict", "train"))
    if kind == "recover3d":
        top = rng.randint(4, 8)
        n = [1 << max(3, top - rng.randint(0, 2)) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "bc": rng.choice("nnd"),
                "wavelet": rng.choice(("cdf3.7", "cdf3.7", "cdf3.5")),
                "vout": rng.random() < 0.25}
    if kind == "recover2d":
        return {"kind": kind, "nx": 1 << rng.randint(5, 10), "ny": 1 << rng.randint(5, 10)}
    if kind == "batch":
        return {"kind": kind, "count": _log_int(rng, 4, 64), "mix": rng.randint(0, 999)}
    if kind in ("solids", "geometry"):
        top = _log_int(rng, 24, 160)
        n = [max(16, int(top * rng.uniform(0.5, 1.0))) for _ in range(3)]
        c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "spheres": rng.randint(1, 8)}
        if kind == "solids":
            c["bc"] = rng.choice("nnd")
            c["method"] = rng.choice(("pcg", "pcg", "vcycles"))
        return c
    if kind == "sweep":
        if rng.random() < 0.5:
            top = rng.randint(4, 8)
            n = [1 << max(3, top - rng.randint(0, 1)) for _ in range(3)]
        else:
            n = [_log_int(rng, 16, 200) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "bc": rng.choice("nnd"),
                "dtype": "f64" if max(n) <= 128 and rng.random() < 0.4 else "f32"}
    factor = rng.choice((1, 2, 4))
    net = [4 * rng.randint(4, 12 if kind == "train" else 16) for _ in range(3)]
    return {"kind": kind, "nx": factor * net[0], "ny": factor * net[1], "nz": factor * net[2],
            "factor": factor}


# ---- inputs -----------------------------------------------------------------
def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _modes(rng, count, kmax):
    """Wave numbers 1..kmax per axis, log-uniform, amplitudes |k|^(-11/6)."""
    k = np.exp(rng.uniform(0.0, math.log(kmax + 0.999), size=(count, 3))).astype(int)
    k = np.maximum(k, 1)
    a = rng.standard_normal(count) * np.sqrt((k * k).sum(1)) ** (-11.0 / 6.0)
    return k, a, rng.uniform(0.0, 2.0 * np.pi, size=(count, 3))


def _field(rng, coords, fns, kmax, count=32):
    """sum_m a_m f(x) g(y) h(z) on (zs, xs, ys); fns per axis x, y, z: 'sin', 'cos'
    (wall conditions) or 'any' (a phase)."""
    k, a, ph = _modes(rng, count, kmax)

    def axis(d):
        t = torch.from_numpy(coords[d]).cuda()
        arg = math.pi * torch.outer(t, torch.from_numpy(k[:, d].astype(np.float64)).cuda())
        if fns[d] == "sin":
            return torch.sin(arg)
        if fns[d] == "cos":
            return torch.cos(arg)
        return torch.cos(arg + torch.from_numpy(ph[:, d]).cuda())

    X, Y, Z = axis(0), axis(1), axis(2) * torch.from_numpy(a).cuda()
    zx = (Z[:, None, :] * X[None, :, :]).reshape(-1, Z.shape[1])
    return (zx @ Y.T.contiguous()).reshape(Z.shape[0], X.shape[0], Y.shape[0])


def _nodes(n):
    return np.arange(n + 1) / n


def _centres(n):
    return (np.arange(n) + 0.5) / n


def velocity(n, dx, bc, seed, kmax=None):
    """FP64 face velocities: the curl of a smooth random edge potential, whose wall-tangential
    components vanish for bc 'n' (no flux through the walls)."""
    nx, ny, nz = n
    rng = np.random.default_rng(seed)
    kmax = max(2, min(16, min(n) // 4)) if kmax is None else kmax
    own, tan = ("cos", "sin") if bc == "n" else ("any", "any")
    qx = _field(rng, (_centres(nx), _nodes(ny), _nodes(nz)), (own, tan, tan), kmax)
    qy = _field(rng, (_nodes(nx), _centres(ny), _nodes(nz)), (tan, own, tan), kmax)
    qz = _field(rng, (_nodes(nx), _nodes(ny), _centres(nz)), (tan, tan, own), kmax)
    hx, hy, hz = dx
    xv = (qz[:, :, 1:] - qz[:, :, :-1]) / hy - (qy[1:] - qy[:-1]) / hz
    yv = (qx[1:] - qx[:-1]) / hz - (qz[:, 1:, :] - qz[:, :-1, :]) / hx
    zv = (qy[:, 1:, :] - qy[:, :-1, :]) / hx - (qx[:, :, 1:] - qx[:, :, :-1]) / hy
    return [t.contiguous() for t in (xv, yv, zv)]


def stream2d(case, seed):
    """A node stream function, zero on the walls: 16 Gaussian vortices."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(_nodes(nx)).cuda()[:, None]
    y = torch.from_numpy(_nodes(ny)).cuda()[None, :]
    psi = torch.zeros((nx + 1, ny + 1), dtype=F64, device="cuda")
    for _ in range(16):
        cx, cy = rng.uniform(0.1, 0.9, 2)
        r, s = rng.uniform(0.02, 0.1), rng.standard_normal()
        psi += s * torch.exp(-((x - cx) ** 2 + (y - cy) ** 2) / (2 * r * r))
    psi[0], psi[-1] = 0, 0
    psi[:, 0], psi[:, -1] = 0, 0
    return psi


def spheres(case, seed):
    """Centres and radii inside the case's box of cubic cells, longest side 1."""
    n = np.array(_dims(case), dtype=np.float64)
    ext = n / n.max()
    rng = np.random.default_rng(seed + 77)
    c = rng.uniform(0.2, 0.8, size=(case.get("spheres", 8), 3)) * ext
    r = rng.uniform(0.05, 0.15, size=len(c)) * ext.min()
    return c, r


def distance(case, centres, radii):
    """FP64 signed distance to the union of the spheres at the cell centres."""
    nx, ny, nz = _dims(case)
    h = 1.0 / max(nx, ny, nz)
    x, y, z = (torch.from_numpy((np.arange(n) + 0.5) * h).cuda() for n in (nx, ny, nz))
    out = torch.full((nz, nx, ny), math.inf, dtype=F64, device="cuda")
    for c, r in zip(centres, radii):
        d = ((z - c[2]) ** 2)[:, None, None] + ((x - c[0]) ** 2)[None, :, None] \
            + ((y - c[1]) ** 2)[None, None, :]
        out = torch.minimum(out, torch.sqrt(d) - r)
    return out


def fractions(ls, h):
    """Wet face fractions (x, y, z faces) of a cell level set, cubic cells of side h."""
    out = []
    for d in (1, 2, 0):
        n = ls.shape[d]
        lo = torch.cat((ls.narrow(d, 0, 1), ls), d)
        hi = torch.cat((ls, ls.narrow(d, n - 1, 1)), d)
        w = torch.sqrt(torch.clamp(h * h - (hi - lo) ** 2, min=1e-14))
        out.append((1.0 - torch.clamp((1.0 - (hi + lo) / w) * 0.5, 0.0, 1.0)).contiguous())
    return out


def solid_inputs(case, seed):
    """FP32 velocity and face fractions of the solid-obstacle step."""
    n = _dims(case)
    h = 1.0 / max(n)
    a = fractions(distance(case, *spheres(case, seed)), h)
    u = velocity(n, (h, h, h), case["bc"], seed, kmax=min(12, max(2, min(n) // 4)))
    return [t.float() for t in u], [t.float() for t in a]


def network_weights():
    """(FP32 parameters, output scale) of the trained network."""
    with open(WEIGHTS, "rb") as fh:
        raw = fh.read()
    count = int(np.frombuffer(raw[8:16], "<u8")[0])
    return (np.frombuffer(raw[32:32 + 4 * count], "<f4").copy(),
            float(np.frombuffer(raw[16:24], "<f8")[0]))


def network_inputs(case, seed):
    """FP32 right-hand side, level set and pressure of one solid-obstacle problem."""
    n = _dims(case)
    rng = np.random.default_rng(seed)
    ls = distance(case, *spheres(case, seed))
    cells = [_centres(v) for v in n]
    f = _field(rng, cells, ("cos", "cos", "cos"), 12) * 50.0
    f = torch.where(ls > 0, f, torch.zeros_like(f))
    p = _field(rng, cells, ("cos", "cos", "cos"), 4) * 0.1
    return f.float(), ls.float(), p.float()


# ---- what a program holds before the call ---------------------------------------
def _shapes(n):
    nx, ny, nz = n
    return [(nz + 1, nx, ny + 1), (nz + 1, nx + 1, ny), (nz, nx + 1, ny + 1)]


def _wavelets(case):
    c, d = PAIRS[case["wavelet"]]
    return W.WaveletType[c], W.WaveletType[d]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "recover3d":
        n = _dims(case)
        dx = tuple(1.0 / v for v in n)
        s["v"] = [t.float() for t in velocity(n, dx, case["bc"], seed)]
        s["q"] = [torch.empty(sh, device="cuda") for sh in _shapes(n)]
        s["vo"] = [torch.empty_like(t) for t in s["v"]] if case["vout"] else []
        s["rec"] = W.CuWaveletPotentialRecover3D(n, dx, case["bc"], *_wavelets(case))
    elif kind == "recover2d":
        nx, ny = case["nx"], case["ny"]
        psi = stream2d(case, seed)
        s["v"] = [((psi[:, 1:] - psi[:, :-1]) * ny).float().contiguous(),
                  (-(psi[1:] - psi[:-1]) * nx).float().contiguous()]
        s["q"] = torch.empty((nx + 1, ny + 1), device="cuda")
        s["rec"] = W.CuWaveletPotentialRecover2D((nx, ny), (1.0 / nx, 1.0 / ny), "n",
                                                 W.WaveletType.WT_CDF3_7, W.WaveletType.WT_CDF4_6)
    elif kind == "batch":
        grids = batch_grids(case)
        dxs = [(1.0 / max(g),) * 3 for g in grids]
        b = W.CuBatchRecover3D(grids, dxs, "n", W.WaveletType.WT_CDF3_7, W.WaveletType.WT_CDF4_6)
        for i, (g, dx) in enumerate(zip(grids, dxs)):
            a = b.arrays(i)
            for key, v in zip(("xv", "yv", "zv"), velocity(g, dx, "n", seed * 1000 + i)):
                a[key].copy_(v)
        b.Capture()
        b.Autotune(2)
        s["rec"] = b
    elif kind == "solids":
        n = _dims(case)
        h = 1.0 / max(n)
        s["n"], s["dx"] = n, (h, h, h)
        s["u0"], s["a"] = solid_inputs(case, seed)
        s["u"] = [torch.empty_like(t) for t in s["u0"]]
        s["mg"] = W.CuMultigridFrac3D(*s["a"], n, s["dx"], case["bc"])
        s["f"], s["p"], s["p_lo"] = (torch.empty((n[2], n[0], n[1]), device="cuda")
                                     for _ in range(3))
    elif kind == "geometry":
        n = _dims(case)
        h = 1.0 / max(n)
        nx, ny, nz = n
        s["n"], s["h"] = n, h
        s["centres"], s["radii"] = spheres(case, seed)
        s["ls"] = W.CuSolidLevelSet3D(n, (h, h, h))
        s["a"] = [torch.empty(sh, device="cuda") for sh in
                  ((nz, nx + 1, ny), (nz, nx, ny + 1), (nz + 1, nx, ny))]
    elif kind == "sweep":
        n = _dims(case)
        dt = F64 if case["dtype"] == "f64" else torch.float32
        dx = tuple(1.0 / max(n) for _ in n)
        s["v"] = [t.to(dt) for t in velocity(n, dx, case["bc"], seed)]
        s["q"] = [torch.empty(sh, dtype=dt, device="cuda") for sh in _shapes(n)]
        s["sweep"] = W.CuParallelSweep3D(n, dx, case["bc"], dtype=dt)
    else:
        n = _dims(case)
        s["f"], s["ls"], s["p"] = network_inputs(case, seed)
        s["p0"] = torch.empty_like(s["f"])
        s["net"] = W.UNet3D(n, seed=1, factor=case["factor"])
        params, scale = network_weights()
        s["net"].set_params(params)
        s["net"].set_output_scale(scale)
    return s


def batch_grids(case):
    r = random.Random(case["mix"])
    return [r.choice(BATCH_GRIDS) for _ in range(case["count"])]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "recover3d":
        s["rec"].Solve(*s["q"], *s["vo"], *s["v"])
        return {"q": s["q"], "v": s["vo"]}
    if kind == "recover2d":
        s["rec"].Solve(s["q"], *s["v"])
        return s["q"]
    if kind == "batch":
        s["rec"].Replay()
        return s["rec"].arena
    if kind == "solids":
        # the step's velocity, then f = -div(a u), p, u <- a (u - grad p)
        for t, t0 in zip(s["u"], s["u0"]):
            t.copy_(t0)
        n, dx, bc = s["n"], s["dx"], case["bc"]
        W.CuConvergence.GetInstance().GetB_3d_frac_vel(s["f"], *s["u"], *s["a"], n, dx, bc)
        if case["method"] == "pcg":
            s["mg"].SolvePCG(s["p"], s["p_lo"], None, s["f"], 1e-6, 100)
        else:
            s["mg"].SolveToTolerance(s["p"], s["p_lo"], None, s["f"], 1e-6, 200)
        W.CuGradient.GetInstance().SubtractGradient3D_Frac_P2(*s["u"], s["p"], s["p_lo"], *s["a"],
                                                              n, dx, bc)
        return s["u"]
    if kind == "geometry":
        ls, h = s["ls"], s["h"]
        ls.InitLsSpheres(s["centres"], s["radii"])
        # exact near the solids, relaxed from far away elsewhere
        ls.ls.masked_fill_(ls.ls > 2 * h, 4.0)
        W.CuFastSweeping.GetInstance().Solve(ls.ls, s["n"], h, 2 * max(s["n"]))
        ls.GetFrac(*s["a"])
        return {"ls": ls.ls, "a": s["a"]}
    if kind == "sweep":
        s["sweep"].Solve(*s["q"], *s["v"])
        s["sweep"].Project(*s["q"])
        return s["q"]
    if kind == "predict":
        s["net"].predict(s["p0"], s["f"], s["ls"], 1.0)
        return s["p0"]
    loss = s["net"].loss_grad(s["f"], s["ls"], s["p"], 1.0)
    s["net"].adam(1e-4)
    return {"loss": loss, "grad": s["net"].get_params(1)}


# ---- FP64 restatements ----------------------------------------------------------
def _faces(n):
    nx, ny, nz = n
    return (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)


def _edges(n):
    return sum(math.prod(sh) for sh in _shapes(n))


# (channels in, channels out, level) of the network's convolutions
LAYERS = ((16, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2),
          (96, 32, 1), (32, 32, 1), (48, 16, 0), (16, 16, 0), (16, 16, 0))


def work(case):
    """Each input read once, each output written once; operations of the definition."""
    kind = case["kind"]
    if kind in ("recover3d", "batch"):
        grids = [_dims(case)] if kind == "recover3d" else batch_grids(case)
        # about 10 operations a sample and line pass, 20 a cell for the projection
        vel, pot = (sum(f(g) for g in grids) for f in (_faces, _edges))
        twice = 2 if case.get("vout") else 1
        return {"bytes": 4.0 * (twice * vel + pot),
                "flops": 30.0 * (twice * vel + pot) + 20.0 * sum(math.prod(g) for g in grids)}
    if kind == "recover2d":
        v = case["nx"] * case["ny"]
        return {"bytes": 12.0 * v, "flops": 80.0 * v}
    n = _dims(case)
    cells = math.prod(n)
    if kind == "solids":
        # velocity in and out, fractions in; ten V-cycles' stencils at the least
        return {"bytes": 4.0 * 3 * _faces(n), "flops": 10 * 8 * 14.0 * cells}
    if kind == "geometry":
        return {"bytes": 4.0 * (cells + _faces(n)), "flops": 2 * max(n) * 20.0 * cells}
    if kind == "sweep":
        size = 8 if case["dtype"] == "f64" else 4
        return {"bytes": float(size * (_faces(n) + _edges(n))),
                "flops": (6 * 2.5 * sum(math.log2(v) for v in n) / 3 + 30.0) * cells}
    net = cells / case["factor"] ** 3
    conv = sum(2.0 * 27 * ci * co * net / 8 ** lv for ci, co, lv in LAYERS)
    if kind == "predict":
        return {"bytes": 12.0 * cells, "flops": conv}
    return {"bytes": 12.0 * cells, "flops": 3 * conv}


def _gradient(p, a, h, bc):
    """Face gradients of the cell field p, zero on dry faces; walls closed ('n') or
    with a zero value on the wall face ('d')."""
    out = []
    for d, af in zip((1, 2, 0), a):
        n = p.shape[d]
        g = torch.zeros_like(af)
        g.narrow(d, 1, n - 1).copy_((p.narrow(d, 1, n - 1) - p.narrow(d, 0, n - 1)) / h)
        if bc == "d":
            g.narrow(d, 0, 1).copy_(p.narrow(d, 0, 1) / (0.5 * h))
            g.narrow(d, n, 1).copy_(-p.narrow(d, n - 1, 1) / (0.5 * h))
        out.append(torch.where(af > 1e-12, g, torch.zeros_like(g)))
    return out


def _minus_div(u, a, h):
    out = 0.0
    for d, uf, af in zip((1, 2, 0), u, a):
        t = uf * af
        n = t.shape[d] - 1
        out = out - (t.narrow(d, 1, n) - t.narrow(d, 0, n)) / h
    return out


def _exact_solids(case, seed):
    """Conjugate gradients (diagonal scaling) in FP64 far below the step's tolerance."""
    u, a = solid_inputs(case, seed)
    u, a = [t.double() for t in u], [t.double() for t in a]
    h, bc = 1.0 / max(_dims(case)), case["bc"]
    f = _minus_div(u, a, h)
    diag = torch.zeros_like(f)
    for d, af in zip((1, 2, 0), a):
        n = f.shape[d]
        w = torch.where(af > 1e-12, af, torch.zeros_like(af)) / (h * h)
        w.narrow(d, 0, 1).mul_(2.0 if bc == "d" else 0.0)
        w.narrow(d, n, 1).mul_(2.0 if bc == "d" else 0.0)
        diag += w.narrow(d, 0, n) + w.narrow(d, 1, n)
    inv = torch.where(diag > 0, 1.0 / torch.clamp(diag, min=1e-300), torch.zeros_like(diag))
    p, r = torch.zeros_like(f), f * (diag > 0)
    z = inv * r
    q, rz = z.clone(), (r * z).sum()
    stop = 1e-11 * float(f.norm())
    for i in range(6000):
        aq = _minus_div(_gradient(q, a, h, bc), a, h)
        alpha = rz / (q * aq).sum()
        p += alpha * q
        r -= alpha * aq
        if i % 25 == 24 and float(r.norm()) <= stop:
            break
        z = inv * r
        new = (r * z).sum()
        q = z + (new / rz) * q
        rz = new
    g = _gradient(p, a, h, bc)
    return [af * (uf - gf) for uf, af, gf in zip(u, a, g)]


def _exact_geometry(case, seed):
    n = _dims(case)
    h = 1.0 / max(n)
    c, r = spheres(case, seed)
    v = distance(case, c.astype(np.float32).astype(np.float64),
                 r.astype(np.float32).astype(np.float64))
    v = torch.where(v > 2 * h, torch.full_like(v, 4.0), v)
    for _ in range(2 * max(n)):
        m = []
        for d in (0, 1, 2):
            wall = torch.full_like(v.narrow(d, 0, 1), 1e8)
            k = v.shape[d] - 1
            m.append(torch.minimum(torch.cat((wall, v.narrow(d, 0, k)), d),
                                   torch.cat((v.narrow(d, 1, k), wall), d)))
        lo, hi = torch.minimum(m[0], m[1]), torch.maximum(m[0], m[1])
        t = torch.maximum(lo, m[2])
        a, b, e = torch.minimum(lo, m[2]), torch.minimum(hi, t), torch.maximum(hi, t)
        u1 = a + h
        u2 = 0.5 * (a + b + torch.sqrt(torch.clamp(2 * h * h - (a - b) ** 2, min=0)))
        u3 = (a + b + e + torch.sqrt(torch.clamp(3 * h * h - (a - b) ** 2 - (a - e) ** 2
                                                 - (b - e) ** 2, min=0))) / 3
        u = torch.where(u1 > b, torch.where(u2 > e, u3, u2), u1)
        v = torch.where(v > -1e-12, u, v)
    return {"ls": v, "a": fractions(v, h)}


def _sine_solve(b, dx):
    """phi with (-L_h) phi = b, zero one node outside, by dense sine transforms."""
    lam, mats = [], []
    for d, h in zip((0, 1, 2), (dx[2], dx[0], dx[1])):
        n = b.shape[d]
        k = torch.arange(1, n + 1, dtype=F64, device="cuda")
        mats.append(math.sqrt(2.0 / (n + 1)) * torch.sin(math.pi / (n + 1) * torch.outer(k, k)))
        lam.append((2.0 * torch.sin(math.pi * k / (2 * (n + 1))) / h) ** 2)

    def along(t):
        for d, S in enumerate(mats):
            t = torch.movedim(t, d, -1)
            t = torch.movedim((t.reshape(-1, t.shape[-1]) @ S).reshape(t.shape), -1, d)
        return t.contiguous()

    return along(along(b) / (lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :]))


def _exact_sweep(case, seed):
    n = _dims(case)
    h = 1.0 / max(n)
    dt = F64 if case["dtype"] == "f64" else torch.float32
    xv, yv, zv = (t.to(dt).double() for t in velocity(n, (h, h, h), case["bc"], seed))
    qx, qy, qz = (torch.zeros(sh, dtype=F64, device="cuda") for sh in _shapes(n))
    qx[1:] = torch.cumsum(yv, 0) * h
    if case["bc"] == "n":
        qy[1:] = -torch.cumsum(xv, 0) * h
        qz[-1, 1:] = -torch.cumsum(qx[-1], 0)
        qx[-1], qy[-1] = 0, 0
        b = -((qx[1:-1, 1:, 1:-1] - qx[1:-1, :-1, 1:-1])
              + (qy[1:-1, 1:-1, 1:] - qy[1:-1, 1:-1, :-1])
              + (qz[1:, 1:-1, 1:-1] - qz[:-1, 1:-1, 1:-1])) / h
        phi = torch.nn.functional.pad(_sine_solve(b, (h, h, h)), (1, 1, 1, 1, 1, 1))
    else:
        qy[0, 1:] = torch.cumsum(zv[0], 0) * h
        qy[1:] = qy[0] - torch.cumsum(xv, 0) * h
        b = torch.zeros((n[2] + 1, n[0] + 1, n[1] + 1), dtype=F64, device="cuda")
        b[:, 1:-1, :] -= (qx[:, 1:, :] - qx[:, :-1, :]) / h
        b[:, :, 1:-1] -= (qy[:, :, 1:] - qy[:, :, :-1]) / h
        b[1:-1] -= (qz[1:] - qz[:-1]) / h
        phi = _sine_solve(b, (h, h, h))
    qx -= (phi[:, 1:, :] - phi[:, :-1, :]) / h
    qy -= (phi[:, :, 1:] - phi[:, :, :-1]) / h
    qz -= (phi[1:] - phi[:-1]) / h
    return [qx, qy, qz]


def _conv3(x, w, bias):
    """3x3x3 convolution of (Z, X, Y, ci) with w (co, 27, ci), zero padding."""
    Z, X, Y, ci = x.shape
    t = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = bias
    for tap in range(27):
        a, b, c = tap // 9, tap // 3 % 3, tap % 3
        sh = t[a:a + Z, b:b + X, c:c + Y].reshape(-1, ci)
        out = out + sh @ w[:, tap].T
    return out.reshape(Z, X, Y, -1)


def _network(params, f, ls, factor):
    """Output of the U-Net on the block means of f and ls, and rms(f) there."""
    def means(t):
        z, x, y = (v // factor for v in t.shape)
        return t.reshape(z, factor, x, factor, y, factor).mean((1, 3, 5))

    off, wb = 0, []
    for ci, co, _ in LAYERS:
        w = params[off:off + co * 27 * ci].reshape(co, 27, ci)
        wb.append((w, params[off + co * 27 * ci:off + co * 27 * ci + co]))
        off += co * (27 * ci + 1)

    def layer(i, *xs):
        y = _conv3(torch.cat(xs, -1) if len(xs) > 1 else xs[0], *wb[i])
        return torch.relu(y) if i < 10 else y[..., 0]

    def pool(t):
        z, x, y, c = t.shape
        return t.reshape(z // 2, 2, x // 2, 2, y // 2, 2, c).mean((1, 3, 5))

    def up(t):
        for d in (0, 1, 2):
            t = t.repeat_interleave(2, d)
        return t

    f, ls = means(f), means(ls)
    rms = f.square().mean().sqrt()
    x = torch.zeros(f.shape + (16,), dtype=F64, device="cuda")
    x[..., 0], x[..., 1] = f / rms, ls
    e0 = layer(1, layer(0, x))
    e1 = layer(3, layer(2, pool(e0)))
    b = layer(5, layer(4, pool(e1)))
    d1 = layer(7, layer(6, up(b), e1))
    return layer(10, layer(9, layer(8, up(d1), e0))), rms, means


def _exact_network(case, seed):
    f, ls, p = (t.double() for t in network_inputs(case, seed))
    params, scale = network_weights()
    w = torch.from_numpy(params).cuda().double()
    if case["kind"] == "predict":
        with torch.no_grad():
            out, rms, _ = _network(w, f, ls, case["factor"])
            for d in range(3):
                n, k = out.shape[d], case["factor"]
                t = (torch.arange(n * k, dtype=F64, device="cuda") + 0.5) / k - 0.5
                t = torch.clamp(t, 0, n - 1)
                i0 = t.floor().long()
                i1 = torch.clamp(i0 + 1, max=n - 1)
                sh = [1, 1, 1]
                sh[d] = -1
                wt = (t - i0).reshape(sh)
                out = out.index_select(d, i0) * (1 - wt) + out.index_select(d, i1) * wt
            return out * rms * scale
    w.requires_grad_(True)
    out, rms, means = _network(w, f, ls, case["factor"])
    e = out - means(p) / (rms * scale)
    loss = (e - e.mean()).square().mean()
    loss.backward()
    return {"loss": float(loss), "grad": w.grad}


def exact(case, seed):
    kind = case["kind"]
    if kind == "recover3d":
        if not case["vout"]:
            return None
        n = _dims(case)
        v = velocity(n, tuple(1.0 / k for k in n), case["bc"], seed)
        return {"q": [None] * 3, "v": [t.float().double() for t in v]}
    if kind == "recover2d":
        return stream2d(case, seed)
    if kind == "batch":
        return None
    if kind == "solids":
        return _exact_solids(case, seed)
    if kind == "geometry":
        return _exact_geometry(case, seed)
    if kind == "sweep":
        return _exact_sweep(case, seed)
    return _exact_network(case, seed)
