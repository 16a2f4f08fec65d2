"""The work this framework is timed on: right-hand sides, whole runs and a serving queue.

A case is one of three kinds:

- "rhs": one right-hand side on the caller's own device buffers (nuc_rhs_noalloc), a
  coupled solver's call; the state is a torch tensor on the GPU.
- "run": a run of one box from a given state: upload, `steps` TVD-RK3 steps on the
  resident state, the state back for a restart file (Context).
- "serve": a queue of small independent boxes handed to the serving loop together, with
  every job's final state fetched (Server).

exact() is the same mathematics in plain torch, FP64, written from the schemes' formulas.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("nuc3d-cartisian_amd"))
import nuc3d_amd as G  # noqa: E402

GAMMA, PRANDTL, T_REF, T_INF = 1.4, 0.72, 110.4, 288.0
SCHEME = {"weno5js": G.WENO5JS, "weno5z": G.WENO5Z, "weno7js": G.WENO7JS, "crweno5": G.CRWENO5, "hccs": G.HCCS}
VIS = {"cd6": G.CD6, "cd8": G.CD8}
RIEMANN = {"lf": G.LF, "ausm": G.AUSM, "ausmp": G.AUSMP}
PRECISION = {"fp64": G.FP64, "mixed": G.MIXED, "fp32": G.FP32}
#: floating operations of one cell's right-hand side (3 directions, 5 variables, 2 signs; viscous terms)
FLOPS = {"weno5js": 2300, "weno5z": 2500, "weno7js": 5200, "crweno5": 3300, "hccs": 4300}


def _box(name, kind, nx, ny, nz, scheme, riemann="lf", vis="cd6", precision="fp64", steps=1, graph=False, field="hit",
         mach=0.1, reynolds=1600.0, cfl=0.5, forced=False):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, scheme=scheme, riemann=riemann, vis=vis,
                precision=precision, steps=steps, graph=graph, field=field, mach=mach, reynolds=reynolds, cfl=cfl,
                forced=forced)


def listed():
    hit = dict(mach=0.3 / math.sqrt(3.0), reynolds=200.0)
    shu = dict(field="shock", mach=1.0 / math.sqrt(1.4), reynolds=2000.0, cfl=0.4)
    return [
        # the smallest call: a coupled solver or a parameter study asks for one right-hand side of a small box
        _box("rhs_32", "rhs", 32, 32, 32, "weno5js"),
        # the same on a ragged box, compact scheme and 8th-order viscous terms
        _box("rhs_97x60x83", "rhs", 97, 60, 83, "crweno5", vis="cd8", mach=0.3),
        # the Taylor-Green configuration at its own size: a long run of short steps, replayed as one graph a step
        _box("run_64_weno5js_graph", "run", 64, 64, 64, "weno5js", steps=100, graph=True, field="tgv"),
        # a box whose lines fit no power of two, compact scheme, default viscous terms
        _box("run_150x132x108_crweno5", "run", 150, 132, 108, "crweno5", steps=30, mach=0.3, reynolds=800.0),
        # the 7th-order scheme with the AUSM+ splitting, 160 cells a side
        _box("run_160_weno7_ausmp", "run", 160, 160, 160, "weno7js", riemann="ausmp", steps=10, **hit),
        # the shock configuration: Shu-Osher profile, long lines in x only
        _box("run_512x128x128_weno5z_ausm", "run", 512, 128, 128, "weno5z", riemann="ausm", steps=20, **shu),
        # decaying turbulence, the benchmark's configuration, in the three precisions a user picks from
        _box("run_256_crweno5", "run", 256, 256, 256, "crweno5", vis="cd8", steps=30, **hit),
        _box("run_256_crweno5_mixed", "run", 256, 256, 256, "crweno5", vis="cd8", precision="mixed", steps=30, **hit),
        _box("run_192_crweno5_fp32", "run", 192, 192, 192, "crweno5", vis="cd8", precision="fp32", steps=24, **hit),
        # the largest: forced turbulence on 512^3, compact hybrid scheme, AUSM, spectral forcing
        _box("run_512_hccs_ausm_forced", "run", 512, 512, 512, "hccs", riemann="ausm", steps=3, forced=True,
             mach=0.5 / math.sqrt(3.0), reynolds=200.0),
        # a queue of uneven small jobs for the serving loop, 24 to 96 cells a side, its three schemes in turn
        dict(name="serve_18", kind="serve", jobs=18, nmin=24, nmax=96, steps=12, draw=20261202),
    ]


def draw(rng):
    """One more case: boxes from 24^3 to 2^24 cells over their logarithm, sides uneven, every kind and option."""
    kind = rng.choice(["rhs", "run", "run", "run", "serve"])
    if kind == "serve":
        nmin = rng.randrange(20, 40)
        return dict(kind="serve", jobs=rng.randrange(6, 21), nmin=nmin, nmax=nmin + rng.randrange(20, 70),
                    steps=rng.randrange(6, 16), draw=rng.randrange(1 << 30))
    top = math.log(2.0 ** (20 if kind == "rhs" else 24))
    side = math.exp(rng.uniform(math.log(24.0 ** 3), top) / 3.0)
    ax, ay = (math.exp(rng.uniform(-0.4, 0.4)) for _ in range(2))
    n = [max(16, min(512, int(round(s)))) for s in (side * ax, side * ay, side / (ax * ay))]
    if rng.random() < 0.5:
        n = [max(16, 16 * round(k / 16)) for k in n]
    while n[0] * n[1] * n[2] > 2 ** (20 if kind == "rhs" else 24):
        n[n.index(max(n))] -= 1
    cells = n[0] * n[1] * n[2]
    scheme = rng.choice(["weno5js", "weno5z", "crweno5", "crweno5", "hccs", "weno7js"])
    precision = "fp64" if kind == "rhs" else rng.choice(["fp64", "fp64", "mixed", "fp32"])
    if precision == "fp32" and scheme == "hccs":
        precision = "mixed"
    forced = kind == "run" and precision != "fp32" and rng.random() < 0.15
    steps = 1 if kind == "rhs" else max(2, min(10 if scheme in ("hccs", "weno7js") else 40, (1 << 28) // cells))
    c = _box("", kind, n[0], n[1], n[2], scheme, rng.choice(["lf", "lf", "ausm", "ausmp"]), rng.choice(["cd6", "cd8"]),
             precision, steps, kind == "run" and cells <= 1 << 19, "hit", round(rng.uniform(0.1, 0.5), 3),
             round(math.exp(rng.uniform(math.log(200.0), math.log(3200.0))), 1), 0.5, forced)
    del c["name"]
    return c


# ---- inputs ----------------------------------------------------------------------------

def _lengths(c):
    """Box lengths: cubic cells, the longest side 2 pi (10 for the shock)."""
    top = max(c["nx"], c["ny"], c["nz"])
    return tuple((10.0 if c["field"] == "shock" else 2 * math.pi) * c[k] / top for k in ("nx", "ny", "nz"))


def _config(c):
    forcing = dict(forcing=G.FORCING_CONST, forcing_k=1.5, forcing_amp=0.05, forcing_amp_hel=0.0) if c["forced"] else {}
    return G.make_config(n=(c["nx"], c["ny"], c["nz"]), L=_lengths(c), scheme=SCHEME[c["scheme"]], vis=VIS[c["vis"]],
                         riemann=RIEMANN[c["riemann"]], precision=PRECISION[c["precision"]], mach=c["mach"],
                         reynolds=c["reynolds"], cfl=c["cfl"], **forcing)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _state(c, seed):
    """The conserved state (5, nz, ny, nx), FP64: a solenoidal velocity of seeded large-scale
    modes over the case's base flow, density and pressure each 1 % uneven."""
    dev, n = _device(), (c["nx"], c["ny"], c["nz"])
    rng = np.random.default_rng(seed)
    L = _lengths(c)
    x = [torch.arange(n[d], dtype=torch.float64, device=dev).add_(0.5).mul_(2 * math.pi / n[d]) for d in range(3)]

    def mode(k, phase, amp):
        """amp[m] cos(k.x + phase) of each of amp's fields, added up over the calls."""
        e = [torch.exp(1j * k[d] * x[d]) for d in range(3)]
        yz = e[2][:, None] * e[1][None, :] * complex(math.cos(phase), math.sin(phase))
        w = (yz[:, :, None] * e[0][None, None, :]).real
        for f, a in amp:
            f.add_(w, alpha=float(a))

    vel = torch.zeros((3,) + n[::-1], dtype=torch.float64, device=dev)
    rho, p = torch.zeros(n[::-1], dtype=torch.float64, device=dev), torch.zeros(n[::-1], dtype=torch.float64, device=dev)
    for i in range(14):
        # three modes of the shell that the forcing acts on, then any
        k = rng.permutation([1, -1, 0]) if i < 3 else rng.integers(-4, 5, 3)
        if not k.any():
            k[0] = 1
        kp = 2 * math.pi * k / np.array(L)   # solenoidal in the box's own lengths
        a = np.cross(kp, rng.standard_normal(3))
        a *= (1.0 + np.sum(k * k)) ** -0.5 / max(1e-9, np.linalg.norm(a))
        b = 0.004 * rng.standard_normal(2)
        mode(k, rng.uniform(0, 2 * math.pi), [(vel[0], a[0]), (vel[1], a[1]), (vel[2], a[2]), (rho, b[0]), (p, b[1])])
    rms = float(vel.square().sum(0).mean().sqrt())
    if c["field"] == "shock":
        vel.mul_(0.05 * 2.629369 / rms)
        xc = (x[0] / (2 * math.pi) - 0.5) * L[0]
        left = xc < -4.0
        rho = torch.where(left, torch.full_like(xc, 3.857143), 1.0 + 0.2 * torch.sin(5.0 * xc)).expand(n[::-1]) * (1 + rho)
        p = torch.where(left, torch.full_like(xc, 10.33333), torch.ones_like(xc)).expand(n[::-1]) * (1 + p)
        vel[0] += torch.where(left, torch.full_like(xc, 2.629369), torch.zeros_like(xc))
    else:
        if c["field"] == "tgv":
            vel.mul_(0.05 / rms)
            s, co = [torch.sin(t) for t in x], [torch.cos(t) for t in x]
            vel[0] += co[2][:, None, None] * co[1][None, :, None] * s[0][None, None, :]
            vel[1] -= co[2][:, None, None] * s[1][None, :, None] * co[0][None, None, :]
        else:
            vel.mul_(1.0 / rms)
        rho = 1.0 + rho
        p = (1.0 + p) / (GAMMA * c["mach"] ** 2)
    q = torch.empty((5,) + n[::-1], dtype=torch.float64, device=dev)
    q[0] = rho
    q[1:4] = rho * vel
    q[4] = p / (GAMMA - 1.0) + 0.5 * rho * vel.square().sum(0)
    return q


def _jobs(c, seed):
    """The queue's boxes: sizes, Mach and Reynolds numbers fixed by the case, their fields by the seed."""
    r = random.Random(c["draw"])
    for j in range(c["jobs"]):
        n = 2 * int(round(math.exp(r.uniform(math.log(c["nmin"]), math.log(c["nmax"]))) / 2))
        yield _box("", "run", n, n, n, ("weno5js", "weno5z", "crweno5")[j % 3], steps=c["steps"],
                   field=("tgv", "hit")[r.randrange(2)], mach=r.uniform(0.1, 0.5),
                   reynolds=r.uniform(400.0, 3200.0)), 1000 * seed + j


def prepare(case, seed):
    if case["kind"] == "serve":
        jobs = [(_config(c), _state(c, s).cpu().numpy().ravel(), c["steps"]) for c, s in _jobs(case, seed)]
        return {"server": G.Server(max_active=16, pack_cells=4 * 40 ** 3, autotune=True), "jobs": jobs}
    cfg, q = _config(case), _state(case, seed)
    if case["kind"] == "rhs":
        return {"cfg": cfg, "q": q, "rhs": torch.empty_like(q), "dt": torch.empty(1, dtype=torch.float64, device=q.device)}
    q = q.cpu().numpy().ravel()
    ctx = G.Context(cfg)
    ctx.upload(q)
    ctx.autotune()
    if case["graph"]:
        ctx.set_graph(True)
    return {"ctx": ctx, "q": q, "steps": case["steps"]}


def run(state):
    if "server" in state:
        srv = state["server"]
        ids = [srv.submit(cfg, q, steps) for cfg, q, steps in state["jobs"]]
        srv.drain()
        return {"q": [srv.result(j)[0] for j in ids]}
    if "ctx" in state:
        ctx = state["ctx"]
        ctx.upload(state["q"])
        ctx.step_async(state["steps"])
        dt, res, _ = ctx.sync()
        return {"q": ctx.download(), "dt": dt, "res": res}
    rc = G.lib().nuc_rhs_noalloc(ctypes.byref(state["cfg"]), ctypes.c_void_p(state["q"].data_ptr()),
                                 ctypes.c_void_p(state["rhs"].data_ptr()), ctypes.c_void_p(state["dt"].data_ptr()),
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if rc != G.NUC_OK:
        raise G.NucError(rc, G.lib().nuc_last_error(None).decode())
    return {"rhs": state["rhs"], "dt": state["dt"]}


def work(case):
    """A right-hand side reads the state and writes the result. A step reads its state and
    u^n and writes the next state: 320 bytes a cell over the three stages in FP64, half
    that where the state is stored in FP32; a run also takes the state in and gives it back."""
    if case["kind"] == "serve":
        every = [work(c) for c, _ in _jobs(case, 0)]
        return {k: sum(w[k] for w in every) for k in ("bytes", "flops")}
    cells = case["nx"] * case["ny"] * case["nz"]
    flops = FLOPS[case["scheme"]] * cells
    if case["kind"] == "rhs":
        return {"bytes": 80.0 * cells, "flops": flops}
    return {"bytes": (case["steps"] * (160.0 if case["precision"] == "fp32" else 320.0) + 80.0) * cells,
            "flops": 3.0 * case["steps"] * flops}


# ---- the same in plain torch, 64 bits ----------------------------------------------------

def _shift(f, k):
    """Cell m + k's value at m, along the first axis (periodic)."""
    return torch.roll(f, -k, 0)


def _is5(f):
    return [13.0 / 12.0 * (f[j] - 2 * f[j + 1] + f[j + 2]) ** 2 + 0.25 * g ** 2
            for j, g in enumerate((f[0] - 4 * f[1] + 3 * f[2], f[1] - f[3], 3 * f[2] - 4 * f[3] + f[4]))]


def _cand5(f):
    return ((2 * f[0] - 7 * f[1] + 11 * f[2]) / 6, (-f[1] + 5 * f[2] + 2 * f[3]) / 6, (2 * f[2] + 5 * f[3] - f[4]) / 6)


def _mean(w, q):
    return sum(a * b for a, b in zip(w, q)) / sum(w)


def _weno7(f, eps):
    """f: 7 upwind points."""
    s = [f[0] * (547 * f[0] - 3882 * f[1] + 4642 * f[2] - 1854 * f[3]) + f[1] * (7043 * f[1] - 17246 * f[2] + 7042 * f[3])
         + f[2] * (11003 * f[2] - 9402 * f[3]) + 2107 * f[3] * f[3],
         f[1] * (267 * f[1] - 1642 * f[2] + 1602 * f[3] - 494 * f[4]) + f[2] * (2843 * f[2] - 5966 * f[3] + 1922 * f[4])
         + f[3] * (3443 * f[3] - 2522 * f[4]) + 547 * f[4] * f[4],
         f[2] * (547 * f[2] - 2522 * f[3] + 1922 * f[4] - 494 * f[5]) + f[3] * (3443 * f[3] - 5966 * f[4] + 1602 * f[5])
         + f[4] * (2843 * f[4] - 1642 * f[5]) + 267 * f[5] * f[5],
         f[3] * (2107 * f[3] - 9402 * f[4] + 7042 * f[5] - 1854 * f[6]) + f[4] * (11003 * f[4] - 17246 * f[5] + 4642 * f[6])
         + f[5] * (7043 * f[5] - 3882 * f[6]) + 547 * f[6] * f[6]]
    q = [(-3 * f[0] + 13 * f[1] - 23 * f[2] + 25 * f[3]) / 12, (f[1] - 5 * f[2] + 13 * f[3] + 3 * f[4]) / 12,
         (-f[2] + 7 * f[3] + 7 * f[4] - f[5]) / 12, (3 * f[3] + 13 * f[4] - 5 * f[5] + f[6]) / 12]
    tau = (s[0] - s[3]).abs()
    return _mean([c / 35.0 * (1 + (tau / (b + eps)) ** 2) for c, b in zip((1, 12, 18, 4), s)], q)


def _solve(lo, di, hi, rhs):
    """Tridiagonal systems along the first axis; the first row's lo and the last row's hi are 0."""
    n, c, d = di.shape[0], torch.empty_like(di), torch.empty_like(rhs)
    c[0], d[0] = hi[0] / di[0], rhs[0] / di[0]
    for m in range(1, n):
        r = 1.0 / (di[m] - lo[m] * c[m - 1])
        c[m], d[m] = hi[m] * r, (rhs[m] - lo[m] * d[m - 1]) * r
    for m in range(n - 2, -1, -1):
        d[m] -= c[m] * d[m + 1]
    return d


def _faces(scheme, f, positive):
    """Interface values (interface m lies between cells m-1 and m) of one sign's flux along the first axis."""
    n = f.shape[0]
    m = torch.arange(n, device=f.device).reshape((n,) + (1,) * (f.dim() - 1))
    if scheme in ("weno7js", "hccs"):
        w = [_shift(f, k) for k in ((-4, -3, -2, -1, 0, 1, 2) if positive else (3, 2, 1, 0, -1, -2, -3))]
        if scheme == "weno7js":
            return _weno7(w, 1e-20)
        edge, ts, s5 = _weno7(w, 1e-40), 4, w[1:6]
    else:
        s5, ts = [_shift(f, k) for k in ((-3, -2, -1, 0, 1) if positive else (2, 1, 0, -1, -2))], 3
    b, q = _is5(s5), _cand5(s5)
    if scheme in ("weno5js", "crweno5"):
        wt = [1.0 / (1e-6 + s) ** 2 for s in b]
        edge = _mean([c * a for c, a in zip((0.1, 0.6, 0.3), wt)], q)
        if scheme == "weno5js":
            return edge
    if scheme == "weno5z":
        if positive:   # the reference's inner positive sweep reads one point twice (src/weno5z.cpp:80)
            odd = 13.0 / 12.0 * (s5[2] - s5[3]) ** 2 + 0.25 * (3 * s5[2] - 4 * s5[3] + s5[4]) ** 2
            b[2] = torch.where((m >= ts) & (m <= n - ts), odd, b[2])
        tau = (b[2] - b[0]).abs()
        return _mean([c * (1 + (tau / (s + 1e-40)) ** 2) for c, s in zip((0.1, 0.6, 0.3), b)], q)
    # compact rows on ts < m < n - ts, the explicit scheme elsewhere
    if scheme == "crweno5":
        w = [c * a for c, a in zip((0.2, 0.5, 0.3), wt)]
        total = sum(w)
        w = [a / total for a in w]
    else:
        tau = (b[2] - b[0]).abs()
        a = [c * (1 + (tau / (s + 1e-40)) ** 2) for c, s in zip((0.2, 0.5, 0.3), b)]
        total = sum(a)
        w = [t / total for t in a]
    lo, di, hi = (2 * w[0] + w[1]) / 3, (w[0] + 2 * (w[1] + w[2])) / 3, w[2] / 3
    rhs = (w[0] * s5[1] + (5 * (w[0] + w[1]) + w[2]) * s5[2] + (w[1] + 5 * w[2]) * s5[3]) / 6
    if scheme == "hccs":
        theta = 1.0 / (1.0 + (total - 1.0) ** 2)
        up, s = theta > 0.5, (1.0 - theta) / theta
        q7 = (-s5[0] + 19 * s5[1] + 239 * s5[2] + 159 * s5[3] + 4 * s5[4]) / 420
        lo, di, hi, rhs = (torch.where(up, r, l * s + r) for l, r in
                           ((lo, torch.full_like(lo, 2 / 7)), (di, torch.full_like(lo, 4 / 7)), (hi, torch.full_like(lo, 1 / 7)), (rhs, q7)))
    inner = (m > ts) & (m < n - ts)
    zero = torch.zeros_like(lo)
    lo, di, hi, rhs = (torch.where(inner, lo, zero), torch.where(inner, di, zero + 1), torch.where(inner, hi, zero),
                       torch.where(inner, rhs, edge))
    return _solve(lo, di, hi, rhs) if positive else _solve(hi, di, lo, rhs)


def _ddx(f, axis, h, vis):
    co = (3 / 4, -3 / 20, 1 / 60) if vis == "cd6" else (4 / 5, -1 / 5, 4 / 105, -1 / 280)
    return sum(a * (torch.roll(f, -k, axis) - torch.roll(f, k, axis)) for k, a in enumerate(co, 1)) / h


def _force(c, vel):
    """The band forcing's force field: the solenoidal part of the shell 1 < |k| < 2 brought to the energy asked for."""
    n = vel.shape[1:]
    u = torch.fft.fftn(vel, dim=(1, 2, 3)) / vel[0].numel()
    k = [torch.round(torch.fft.fftfreq(s, dtype=torch.float64, device=vel.device) * s) for s in n]
    kv = torch.stack(torch.broadcast_tensors(k[2][None, None, :], k[1][None, :, None], k[0][:, None, None]))
    km = kv.square().sum(0).sqrt()
    k1 = torch.where(km < 1e-6, torch.ones_like(km), km)
    comp = (kv * u).sum(0) / k1 * kv / k1
    sol = u - comp
    band = (k1 - 1.5).abs() < 0.5
    es, ec = (0.5 * (v.abs().square().sum(0) * band).sum() for v in (sol, comp))
    shell = (km - 1.5).abs() < 0.5
    return torch.fft.ifftn((torch.sqrt((0.05 - ec).abs() / es) - 1.0) * sol * shell, dim=(1, 2, 3)).real * vel[0].numel()


def _rhs(c, q):
    """(dQ/dt = -rhs, time step at CFL 1) of the state q (5, nz, ny, nx)."""
    L, n = _lengths(c), (c["nx"], c["ny"], c["nz"])
    h = [L[d] / n[d] for d in range(3)]
    rho, vel = q[0], q[1:4] / q[0]
    p = ((q[4] - 0.5 * rho * vel.square().sum(0)) * (GAMMA - 1.0)).abs()
    cs = torch.sqrt(GAMMA * p / rho)
    lam = [(vel[d].abs() + cs).max() for d in range(3)]
    if c["riemann"] == "lf":   # the y maximum also takes the z eigenvalues, which then do not count (src/physicsModel.cpp:653-654)
        lam = [lam[0], torch.maximum(lam[1], lam[2]), torch.zeros_like(lam[2])]
    dt = 1.0 / sum(a / s for a, s in zip(lam, h))
    r = torch.zeros_like(q)
    # viscous stresses (off-diagonals carry -2/3 div u as the reference has them) and heat flux
    T = GAMMA * c["mach"] ** 2 * p / rho
    g = [[_ddx(vel[i], 2 - d, h[d], c["vis"]) for d in range(3)] for i in range(3)]
    S = T_REF / T_INF
    mu = (1 + S) / (T + S) * T * torch.sqrt(T) / c["reynolds"]
    div = g[0][0] + g[1][1] + g[2][2]
    tau = [[mu * (g[i][d] + g[d][i] - 2.0 / 3.0 * div) for d in range(3)] for i in range(3)]
    k = mu / ((GAMMA - 1.0) * c["mach"] ** 2 * PRANDTL)
    for d in range(3):
        axis = 2 - d
        for i in range(3):
            r[1 + i] -= _ddx(tau[i][d], axis, h[d], c["vis"])
        heat = k * _ddx(T, axis, h[d], c["vis"])
        r[4] -= _ddx(sum(vel[i] * tau[i][d] for i in range(3)) + heat, axis, h[d], c["vis"])
    del g, tau, div, k, mu
    if c["forced"]:
        f = _force(c, vel)
        r[1:4] -= f
        fu = (f * vel).sum(0)
        r[4] += fu.mean() - fu
    for d in range(3):
        axis, ud = 2 - d, vel[d]
        if c["riemann"] == "lf":
            F = ud * q
            F[1 + d] += p
            F[4] += ud * p
            s = (ud.abs() + cs) * q
            split = (0.5 * (F + s), 0.5 * (F - s))
        else:
            mach = ud / cs
            inside = mach.abs() < 1
            a, b, m2 = mach + 1, mach - 1, mach * mach - 1
            mp = torch.where(inside, 0.25 * a ** 2 + 0.125 * m2 ** 2, 0.5 * (mach + mach.abs())) * cs
            mn = torch.where(inside, -0.25 * b ** 2 - 0.125 * m2 ** 2, 0.5 * (mach - mach.abs())) * cs
            if c["riemann"] == "ausmp":
                pp = p * (0.25 * a ** 2 * (2 - mach) + 0.1875 * mach * m2 ** 2)
                pn = p * (0.25 * b ** 2 * (2 + mach) - 0.1875 * mach * m2 ** 2)
            else:
                pp, pn = p * a / 2, -p * b / 2
            out = torch.where(inside, torch.ones_like(mach), mach)
            pp = torch.where(inside, pp, 0.5 * p * (mach + mach.abs()) / out)
            pn = torch.where(inside, pn, 0.5 * p * (mach - mach.abs()) / out)
            split = []
            for ma, pa in ((mp, pp), (mn, pn)):
                F = ma * q
                F[1 + d] += pa
                F[4] += ma * p
                split.append(F)
        total = 0
        for F, positive in zip(split, (True, False)):
            total = total + _faces(c["scheme"], F.movedim(1 + axis, 0).contiguous(), positive)
        r += ((_shift(total, 1) - total) / h[d]).movedim(0, 1 + axis)
    return r, dt


def _advance(c, q):
    """(state after c's steps, the last step's dt and residual)."""
    for _ in range(c["steps"]):
        r, dt = _rhs(c, q)
        dt = dt * c["cfl"]
        a = q - r * dt
        a = 0.75 * q + 0.25 * (a - _rhs(c, a)[0] * dt)
        a = q / 3.0 + 2.0 / 3.0 * (a - _rhs(c, a)[0] * dt)
        q, before = a, q
    return q, dt, ((q - before).square().sum() / q.numel()).sqrt() / dt


def exact(case, seed):
    if case["kind"] == "serve":
        return {"q": [_advance(c, _state(c, s))[0].reshape(-1) for c, s in _jobs(case, seed)]}
    if case["nx"] * case["ny"] * case["nz"] * case["steps"] > 5 << 26:
        return None   # over about 20 seconds
    q = _state(case, seed)
    if case["kind"] == "rhs":
        r, dt = _rhs(case, q)
        return {"rhs": r, "dt": dt.reshape(1)}
    q, dt, res = _advance(case, q)
    return {"q": q.reshape(-1), "dt": float(dt), "res": float(res)}
