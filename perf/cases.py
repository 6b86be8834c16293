"""The work whose speed is measured: what programs that use this framework have
it do, through its public entry points, over the sizes its configurations,
tests and benchmark use.

A case is a dict of plain values:

  kind      "eval"      one vector to one fitness, far field and phase (tomo_eval)
            "noalloc"   the same through tomo_eval_noalloc
            "steps"     one simulation stepped by hand, its fields and far field read
            "batch"     a population of vectors in one call (tomo_eval_batch)
            "requests"  several requests of different grids through the request loop
            "objective" preset + vector to a fitness (tomo_fitness, the FDTD_GPU / FDTD_CPU shims' call)
  physics   "antenna" (physical mode), "ref_gpu" or "ref_cpu" (the reference's two semantics)
  schedule  which of the framework's schedules the program has installed
            ("plain", "batch", "dropin"), or "default": it has installed none
  grid, steps, antennas, freqs, angles, vectors, tumours, dft64

`exact` restates the physics in 64 bits with torch: Yee leapfrog, CPML, the
Debye current, the running transform of the contour and the projection.
"""
import math

import numpy as np
import torch

import tomography_amd as t
from tomography_amd import workloads

SCHEDULES = {"plain": workloads.PLAIN_SCHEDULE, "batch": workloads.BATCH_SCHEDULE, "dropin": workloads.REF_SCHEDULE}
REF_PRESETS = {"ref_gpu": t.PRESET_REF_GPU, "ref_cpu": t.PRESET_REF_CPU}


def _antenna(name, kind, schedule, grid, steps, antennas=1, freqs=8, angles=180, vectors=1, tumours=1, dft64=False):
    return dict(name=name, kind=kind, physics="antenna", schedule=schedule, grid=grid, steps=steps, antennas=antennas,
                freqs=freqs, angles=angles, vectors=vectors, tumours=tumours, dft64=dft64)


def listed():
    return [
        # The smallest use: a program that steps one 128^2 simulation itself and
        # reads its fields between the steps (movies, probes, convergence studies).
        _antenna("steps 128", "steps", "default", 128, 320, 2, 4, 36),
        # One evaluation of the small benchmark grid, as a search that issues its
        # vectors one by one does.
        _antenna("eval 256", "eval", "plain", 256, 2048),
        # A program that has installed no schedule: odd grid, two antennas, two tumours.
        _antenna("eval 363 default", "eval", "default", 363, 2904, 2, tumours=2),
        # The allocation-free entry in a serving loop.
        _antenna("noalloc 512", "noalloc", "plain", 512, 4096),
        # A grid between the powers of two, as the uneven mix has them.
        _antenna("eval 725", "eval", "plain", 725, 5800, tumours=3),
        # The headline workload: one 1024^2 evaluation of 8192 steps.
        _antenna("eval 1024", "eval", "plain", 1024, 8192),
        # One generation of a small search: 16 vectors of a 128^2 phantom, four antennas.
        _antenna("batch 128", "batch", "batch", 128, 800, 4, 4, 36, vectors=16),
        # A part of the 64-vector benchmark population: 16 antennas of 512^2 each.
        _antenna("batch 512", "batch", "batch", 512, 4096, 16, 16, 360, vectors=4),
        # Continuous batching: requests of many grids, one antenna each (the uneven mix).
        _antenna("requests 1448", "requests", "batch", 1448, 0, 1, vectors=12, tumours=3),
        # Continuous batching with several antennas a request (the serving mix).
        _antenna("requests 512", "requests", "batch", 512, 0, 4, vectors=8, tumours=4),
        # The drop-in objective: what a driver of the reference calls for each vector.
        dict(name="objective gpu", kind="objective", physics="ref_gpu", schedule="dropin", grid=401, steps=2000, vectors=1),
        # A population under the reference's CPU semantics (162 parameters), in one call.
        dict(name="batch ref", kind="batch", physics="ref_cpu", schedule="batch", grid=401, steps=2000, vectors=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: The most cell-steps of a drawn case (the 512^2 population has 6.9e10).
MOST = 6.0e10


def draw(rng):
    kind = rng.choice(["eval", "eval", "noalloc", "steps", "batch", "batch", "requests", "objective", "ref batch"])
    if kind == "objective":
        # the shims' configuration is fixed: the preset's grid, of either semantics; a case of its own by its vector
        return dict(kind="objective", physics=rng.choice(["ref_gpu", "ref_cpu"]), schedule="dropin", grid=401, steps=2000,
                    vectors=1, vector=rng.randrange(1 << 20))
    if kind == "ref batch":
        grid = _log_int(rng, 101, 501)
        steps = _log_int(rng, 300, 2000)
        vectors = min(_log_int(rng, 1, 16), max(1, int(MOST / 3 / (4.0 * grid * grid * steps))))
        return dict(kind="batch", physics=rng.choice(["ref_gpu", "ref_cpu"]), schedule=rng.choice(["batch", "dropin", "default"]),
                    grid=grid, steps=steps, vectors=vectors)
    freqs, angles = rng.randint(1, 16), rng.randint(24, 360)
    tumours = rng.randint(1, 4)
    if kind == "steps":
        return {**_antenna("", kind, rng.choice(["default", "plain", "batch"]), _log_int(rng, 96, 512), 32 * rng.randint(4, 20), 2,
                           min(freqs, 8), angles, 1, tumours), "name": "steps drawn"}
    if kind in ("eval", "noalloc"):
        grid = _log_int(rng, 96, 1024)
        steps = min(8192, max(512, int(8 * grid * rng.uniform(0.7, 1.0))))
        antennas = rng.randint(1, 4) if grid < 500 else 1
        schedule = rng.choice(["plain", "plain", "default"])
        return {**_antenna("", kind, schedule, grid, steps, antennas, freqs, angles, 1, tumours, rng.random() < 0.15),
                "name": kind + " drawn"}
    if kind == "batch":
        grid = _log_int(rng, 96, 640)
        antennas, steps = rng.choice([1, 2, 4, 8, 16]), max(400, min(4096, 6 * grid + rng.randint(0, 300)))
        vectors = min(_log_int(rng, 2, 48), max(1, int(MOST / (float(grid) * grid * steps * antennas))))
        return {**_antenna("", kind, rng.choice(["batch", "batch", "default"]), grid, steps, antennas, freqs, angles, vectors, tumours),
                "name": "batch drawn"}
    grid = _log_int(rng, 300, 1448)
    antennas = rng.choice([1, 1, 2, 4]) if grid < 900 else 1
    return {**_antenna("", "requests", rng.choice(["batch", "batch", "default"]), grid, 0, antennas, 8, 180, rng.randint(4, 10), tumours),
            "name": "requests drawn"}


# ---------------------------------------------------------------- inputs
def _config(case, grid=None, steps=None):
    """The configuration of a case (of one of its requests)."""
    if case["physics"] != "antenna":
        cfg = t.preset(REF_PRESETS[case["physics"]])
        if case["grid"] != cfg.nx:  # the contour keeps its place relative to the grid
            cfg = cfg.copy(nx=case["grid"], ny=case["grid"], ntff_offset=max(12, case["grid"] // 4 - 12))
        return cfg.copy(steps=case["steps"])
    n, steps = grid or case["grid"], steps or case["steps"]
    if n < 200:  # the small phantom of a 48..100 mm domain
        cfg = t.preset(t.PRESET_CFG1).copy(nx=n, ny=n, breast_radius=0.14 * n * 1e-3, skin_thickness=0.0015,
                                            src_radius=0.17 * n * 1e-3)
    elif n >= 900 and case["kind"] != "requests":  # the fine grid: 0.25 mm
        cfg = t.preset(t.PRESET_CFG2).copy(nx=n, ny=n)
    else:
        cfg = t.preset(t.PRESET_CFG4, n)
    flags = t.FLAG_DFT_FP64 if case["dft64"] else 0
    return cfg.copy(steps=steps, n_exc=case["antennas"], n_freq=case["freqs"], n_angles=case["angles"], flags=flags)


def _vectors(case, seed):
    rng = np.random.default_rng([seed, case.get("vector", 0)])
    k = case["vectors"]
    if case["physics"] == "ref_gpu":
        return np.concatenate([rng.uniform(1, 7, (k, 9)), rng.uniform(1.5, 41, (k, 9)), rng.uniform(0, 0.3, (k, 9))], axis=1)
    if case["physics"] == "ref_cpu":
        return np.concatenate([rng.uniform(1, 40, (k, 81)), rng.uniform(0, 1.1, (k, 81))], axis=1)
    v = workloads.seeded_vectors(k, 8 * case["tumours"], int(rng.integers(1 << 30)))
    if case["kind"] != "requests" and case["grid"] < 200:
        for b in range(0, v.shape[1], 8):  # inside the small phantom
            v[:, b:b + 2] *= 0.5
            v[:, b + 2] = np.minimum(v[:, b + 2], 4.0)
    return v


def _requests(case, seed):
    """(configuration, vector) of each request: grids log-spaced from a quarter of the largest, in an order of their own."""
    rng = np.random.default_rng(seed)
    k = case["vectors"]
    grids = np.exp(np.linspace(np.log(max(200, case["grid"] // 4)), np.log(case["grid"]), k)).astype(int)
    out = []
    for i in np.random.default_rng(k).permutation(k):  # sizes and order are the case's, vectors the seed's
        g = int(grids[i])
        steps = min(4096, max(2048, 4 * g))
        out.append((_config(case, g, steps), workloads.seeded_vectors(1, 8 * (1 + i % case["tumours"]), int(rng.integers(1 << 30)))[0]))
    return out


def _measurement(case, cfg):
    """The measured far field a reference-compatible evaluation compares with: the packaged one for the preset's own size."""
    kind = "gpu" if case["physics"] == "ref_gpu" else "cpu"
    return t.measurement(kind)[:cfg.farfield_len()]


def prepare(case, seed):
    ctx = t.Context()
    if case["schedule"] != "default":
        ctx.set_schedule(**SCHEDULES[case["schedule"]])
    s = dict(kind=case["kind"], ctx=ctx)
    if case["kind"] == "requests":
        s["requests"] = _requests(case, seed)
        for cfg, _ in s["requests"]:
            ctx.target_farfield(cfg)  # the context keeps the targets of its configurations
        return s
    s["cfg"], s["vectors"] = _config(case), _vectors(case, seed)
    if case["kind"] == "objective":
        s["preset"] = REF_PRESETS[case["physics"]]
    elif case["physics"] != "antenna":
        s["target"] = _measurement(case, s["cfg"])
    elif case["kind"] != "steps":
        s["target"] = ctx.target_farfield(s["cfg"])
    return s


# ---------------------------------------------------------------- one pass
def _far(D, P):
    """Far field and phase as one complex record."""
    return np.sqrt(D) * np.exp(1j * P)


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "eval":
        fit, D, P = ctx.eval(state["cfg"], state["vectors"][0], target=state["target"], want_farfield=True)
        return {"fitness": fit, "far": _far(D, P)}
    if kind == "noalloc":
        fit, D, P = ctx.eval_noalloc(state["cfg"], state["vectors"][0], state["target"], want_farfield=True)
        return {"fitness": fit, "far": _far(D, P)}
    if kind == "batch":
        fit, D = ctx.eval_batch(state["cfg"], state["vectors"], target=state["target"], want_farfield=True)
        return {"fitness": fit, "D": D}
    if kind == "objective":
        return {"fitness": ctx.fitness(state["preset"], state["vectors"][0])}
    if kind == "requests":
        tickets = [ctx.submit(cfg, v) for cfg, v in state["requests"]]
        return {"fitness": np.array([ctx.wait(k)[0] for k in tickets])}
    cfg = state["cfg"]
    sim = ctx.sim(cfg, state["vectors"][0], exc=1)
    try:
        frames = []
        for _ in range(4):
            sim.step(cfg.steps // 4)
            frames.append(sim.fields())
        J, M = sim.dft()
        D, P = sim.farfield()
    finally:
        sim.close()
    return {"frames": frames, "J": J, "M": M, "far": _far(D, P)}


def _cell_steps(case):
    if case["kind"] == "requests":
        return sum(workloads.cell_steps(cfg) for cfg, _ in _requests(case, 0))
    cfg = _config(case)
    return workloads.cell_steps(cfg) * (1.0 / cfg.n_exc if case["kind"] == "steps" else case["vectors"])


def work(case):
    """A cell-step is 12 operations in vacuum (six differences and sums, three
    products with their additions); the state can stay on the chip, so a pass
    has to move the vectors in and the records out."""
    if case["kind"] == "requests":
        moved = sum(8 * v.size + 8 for _, v in _requests(case, 0))
    else:
        cfg = _config(case)
        moved = 8 * _vectors(case, 0).size + 8 * case["vectors"]
        if case["kind"] == "steps":
            moved += 4 * 4 * 4 * (cfg.nx + 1) * (cfg.ny + 1) + 16 * cfg.n_freq * cfg.contour_len() + 8 * cfg.n_freq * cfg.n_angles
        elif case["kind"] != "objective":
            moved += 8 * cfg.farfield_len() * case["vectors"]
    return {"bytes": float(moved), "flops": 12.0 * _cell_steps(case)}


# ---------------------------------------------------------------- 64-bit restatement
EPS0, MU0 = 8.85418e-12, math.pi * 4e-7
C0, ETA0 = 1.0 / math.sqrt(MU0 * EPS0), math.sqrt(MU0 / EPS0)
F32 = np.float32


class _SplitMix:
    def __init__(self, seed):
        self.s = seed & (2 ** 64 - 1)

    def u01(self):
        m = 2 ** 64 - 1
        self.s = (self.s + 0x9E3779B97F4A7C15) & m
        z = self.s
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
        return ((z ^ (z >> 31)) >> 11) / 9007199254740992.0


def _target_vector(cfg):
    r = _SplitMix(cfg.seed ^ 0x7A26E7)
    return np.array([-15.0 + 30.0 * r.u01(), -15.0 + 30.0 * r.u01(), 2.0 + 4.0 * r.u01(), 20.0, 34.0, 13.0, 0.0, 0.0])


def _phantom(cfg, p):
    """Material map (the rasteriser compares in 32 bits) and {eps_inf, delta_eps, tau, sigma} of the materials."""
    ro, ri = cfg.breast_radius, cfg.breast_radius - cfg.skin_thickness
    r = _SplitMix((cfg.seed ^ 0xE111B5E5) + (int(math.floor(p[7])) if p[7] > 0 else 0))
    X = ((np.arange(cfg.nx + 1) - cfg.nx // 2).astype(F32) * F32(cfg.dx))[None, :]
    Y = ((np.arange(cfg.ny + 1) - cfg.ny // 2).astype(F32) * F32(cfg.dy))[:, None]

    def disc(cx, cy, r2):
        dX, dY = X - F32(cx), Y - F32(cy)
        return dX * dX + dY * dY <= F32(r2)
    mats = [(1.0, 0.0, 0.0, 0.0), (36.0, 0.0, 0.0, 4.0), (3.1, 1.6, 13e-12, 0.0), (12.8, 24.6, 13e-12, 0.0)]
    m = np.zeros((cfg.ny + 1, cfg.nx + 1), np.int64)
    m[disc(0, 0, ro * ro)] = 1
    inner = disc(0, 0, ri * ri) & (m == 1)
    m[inner] = 2
    for _ in range(3):
        rho, ph = (ri - 0.012) * math.sqrt(r.u01()), 2 * math.pi * r.u01()
        a, b, th = 0.004 + 0.008 * r.u01(), 0.004 + 0.008 * r.u01(), math.pi * r.u01()
        dX, dY = X - F32(rho * math.cos(ph)), Y - F32(rho * math.sin(ph))
        c, s = F32(math.cos(th)), F32(math.sin(th))
        u, v = dX * c + dY * s, dY * c - dX * s
        m[(u * u * F32(1 / (a * a)) + v * v * F32(1 / (b * b)) <= F32(1)) & inner] = 3
    for k in range(0, min(len(p), 32), 8):
        if not p[k + 2] > 0:
            continue
        rr = min(6.0, max(2.0, p[k + 2])) * 1e-3
        m[disc(p[k] * 1e-3, p[k + 1] * 1e-3, rr * rr) & inner] = len(mats)
        mats.append((p[k + 3], p[k + 4], p[k + 5] * 1e-12, p[k + 6]))
    return m, mats


def _ref_map(cfg, p):
    """Patch map of the reference's disc and the coefficients of each material:
    Ez, curl, the two incident terms, Jp, and the two of the Jp update."""
    n, np_, R, dx, dt = cfg.nx, cfg.numpatches, cfg.breast_radius, cfg.dx, cfg.dt
    i = np.arange(n + 1, dtype=np.float64)
    xc = np.trunc((i - (n // 2 - int(R / dx))) / (2 * R / (np_ * dx))).astype(np.int64)
    yc = np.trunc((i - (n // 2 - R / dx)) / (2 * R / (np_ * dx))).astype(np.int64)
    rad = np.sqrt(((i - n // 2) * dx)[None, :] ** 2 + ((i - n // 2) * dx)[:, None] ** 2).astype(F32)
    m = np.where(rad.astype(np.float64) <= R, 1 + xc[None, :] + np_ * yc[:, None], 0)
    img = np.asarray(p, F32).astype(np.float64)
    n2, rows = np_ * np_, []
    for k in range(1 + n2):
        if cfg.flags & t.FLAG_CPU_COEFS:
            er, sg = (img[k - 1], img[k - 1 + n2]) if k else (1.0, 0.0)
            d = 2 * er * EPS0 + dt * sg
            rows.append(((2 * er * EPS0 - dt * sg) / d, 2 * dt / dx / d, (2 * (EPS0 - EPS0 * er) - sg * dt) / d,
                         -(2 * (EPS0 - EPS0 * er) + sg * dt) / d, 0.0, 0.0, 0.0))
            continue
        ei, de, sg = (img[k - 1], img[k - 1 + n2], img[k - 1 + 2 * n2]) if k else (1.0, 0.0, 0.0)
        tr = cfg.debye_tau
        kp, bp = (1 - dt / (2 * tr)) / (1 + dt / (2 * tr)), EPS0 * de * dt / (tr * (1 + dt / (2 * tr)))
        d = 2 * ei * EPS0 + sg * dt + bp
        rows.append(((2 * ei * EPS0 - sg * dt + bp) / d, 2 * dt / dx / d, (-2 * EPS0 * ei + 2 * EPS0 - sg * dt - bp) / d,
                     (2 * EPS0 * ei - 2 * EPS0 - sg * dt + bp) / d, (1 + kp) * dt / d, kp, bp / dt))
    return m, np.array(rows)


def _profiles(cfg):
    """1/kappa, a, b of the CPML over a line of E nodes (0..n) and of H nodes (0..n-1); identity off the strips."""
    nc, n, dt, dx = cfg.ncpml, cfg.nx, cfg.dt, cfg.dx
    ref = cfg.mode == t.MODE_REF_COMPAT
    out = []
    for h in (0, 1):
        rho = (np.arange(nc) + (0.75 if h else 0.25)) / nc
        g = rho ** cfg.cpml_order
        sig, kap = cfg.sigma_max * g, 1 + (cfg.kappa_max - 1) * g
        al = cfg.alpha_max * (rho if ref else 1 - rho)
        b = np.exp(-(dt / EPS0) * (sig / kap + al))
        den = dx * (sig * kap + al * kap * kap)
        a = sig * (b - 1) / np.where(den == 0, 1, den)
        line = np.zeros((3, n + (0 if h else 1)))
        line[0] = 1.0
        if h:  # H strip cell i sits nc - 1 - i from the low edge, n - nc + i at the high one
            line[:, nc - 1 - np.arange(nc)] = 1 / kap, a, b
            line[:, n - nc + np.arange(nc)] = 1 / kap, a, b
        else:
            line[:, nc - np.arange(nc)] = 1 / kap, a, b
            line[:, n - nc + np.arange(nc)] = 1 / kap, a, b
        out.append(line)
    return out


def _contour(cfg):
    """(x, y, leg) of the contour points: bottom, right, top, left."""
    ref, D, nx, ny = cfg.mode == t.MODE_REF_COMPAT, cfg.ntff_offset, cfg.nx, cfg.ny
    xhi, ylo = (nx - D - 2, D) if ref else (nx - D - 1, D + 1)
    xs, ys = np.arange(D + 1, xhi + 1), np.arange(ylo, ny - D)
    x = np.concatenate([xs, np.full(ys.size, nx - D - 1), xs[::-1], np.full(ys.size, D)])
    y = np.concatenate([np.full(xs.size, D), ys, np.full(xs.size, ny - D - 1), ys[::-1]])
    return x, y, np.repeat([0, 1, 2, 3], [xs.size, ys.size, xs.size, ys.size])


def _frequencies(cfg):
    f = cfg.f_start + (cfg.f_stop - cfg.f_start) / max(1, cfg.n_freq - 1) * np.arange(cfg.n_freq)
    return f.astype(F32).astype(np.float64) if cfg.mode == t.MODE_REF_COMPAT else f


class _Exact:
    """The simulations (vector, excitation) of one configuration, advanced together in 64 bits."""

    def __init__(self, cfg, vectors, excs):
        self.cfg, self.dev = cfg, torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.ref = cfg.mode == t.MODE_REF_COMPAT
        nx, ny, B = cfg.nx, cfg.ny, len(vectors) * len(excs)
        z = lambda *s: torch.zeros(*s, dtype=torch.float64, device=self.dev)  # noqa: E731
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)  # noqa: E731
        maps, rows = [], []
        for p in vectors:
            if self.ref:
                m, r = _ref_map(cfg, p)
            else:
                m, mats = _phantom(cfg, p)
                r = []
                for ei, de, tau, sg in mats:
                    dt = cfg.dt
                    bp = EPS0 * de * dt / (tau * (1 + dt / (2 * tau))) if de > 0 else 0.0
                    kp = (1 - dt / (2 * tau)) / (1 + dt / (2 * tau)) if de > 0 else 0.0
                    d = 2 * ei * EPS0 + sg * dt + bp
                    r.append(((2 * ei * EPS0 - sg * dt + bp) / d, 2 * dt / (cfg.dx * d), 0.0, 0.0, (1 + kp) * dt / d, kp, bp / dt))
                r = np.array(r)
            maps.append(m), rows.append(r)
        # the box of cells that are not vacuum: Jp and the incident terms live there
        some = np.logical_or.reduce([m > 0 for m in maps])
        yy, xx = np.nonzero(some[1:ny, 1:nx])
        self.box = (slice(yy.min(), yy.max() + 1), slice(xx.min(), xx.max() + 1)) if yy.size else (slice(0, 1), slice(0, 1))
        co = np.stack([np.moveaxis(r[m], -1, 0)[:, 1:ny, 1:nx] for m, r in zip(maps, rows)])
        each = lambda k, box=False: T(np.repeat(co[(slice(None), k) + (self.box if box else ())], len(excs), axis=0))  # noqa: E731
        self.ca, self.cb = each(0), each(1)
        self.ceic, self.ceip, self.cj, self.kp, self.bp = (each(k, True) for k in range(2, 7))
        self.ez, self.hx, self.hy = z(B, ny + 1, nx + 1), z(B, ny, nx), z(B, ny, nx)
        self.jp = torch.zeros_like(self.cj)
        self.phx, self.phy, self.pex, self.pey = z(B, ny, nx), z(B, ny, nx), z(B, ny - 1, nx - 1), z(B, ny - 1, nx - 1)
        e, h = _profiles(cfg)
        self.e = [T(v[1:nx]) for v in e]
        self.h = [T(v) for v in h]
        ys = np.zeros(nx - 1, bool)
        ys[:cfg.ncpml] = ys[-cfg.ncpml:] = True
        self.strip = torch.as_tensor(ys, device=self.dev)
        self.n, self.B, self.excs = 0, B, list(excs) * len(vectors)
        # contour samples
        self.x, self.y, self.leg = _contour(cfg)
        ix = lambda a: torch.as_tensor(np.asarray(a, np.int64), device=self.dev)  # noqa: E731
        yf = np.isin(self.leg, (0, 2))
        self.at_h = ix(self.y * nx + self.x)
        self.at_0 = ix(self.y * (nx + 1) + self.x)
        self.at_1 = ix((self.y + yf) * (nx + 1) + self.x + ~yf)
        self.yface = torch.as_tensor(yf, device=self.dev)
        self.freq = _frequencies(cfg)
        P = self.x.size
        self.J = torch.zeros(B, cfg.n_freq, P, dtype=torch.complex128, device=self.dev)
        self.M = torch.zeros_like(self.J)
        self.samples, self.sgn = [], T(np.array([1, 1, -1, -1.0])[self.leg] * float(F32(cfg.dt)))
        if self.ref:
            phi = np.array([k * 2 * math.pi / cfg.n_exc for k in self.excs])
            ox = 0 if cfg.flags & t.FLAG_FWF_ABS_ORIGIN else nx // 2
            X, Y = np.arange(1, nx)[self.box[1]] - ox, np.arange(1, ny)[self.box[0]] - ox
            self.delay = T(-cfg.pulse_t0 - cfg.breast_radius / C0 - np.sin(phi)[:, None, None] * Y[None, :, None] * cfg.dx / C0
                           - np.cos(phi)[:, None, None] * X[None, None, :] * cfg.dx / C0)
        else:
            th = [2 * math.pi * k / cfg.n_exc for k in self.excs]
            rnd = lambda v: int(math.floor(abs(v) + 0.5)) * (1 if v >= 0 else -1)  # noqa: E731
            self.sx = ix([nx // 2 + rnd(cfg.src_radius * math.cos(a) / cfg.dx) for a in th])
            self.sy = ix([ny // 2 + rnd(cfg.src_radius * math.sin(a) / cfg.dx) for a in th])
            self.every = torch.arange(B, device=self.dev)

    def _source(self, n):
        u = ((n + 1) * self.cfg.dt - self.cfg.pulse_t0) / self.cfg.pulse_tau
        return -u * math.exp(-u * u)

    def step(self, count):
        cfg, ez, hx, hy = self.cfg, self.ez, self.hx, self.hy
        (ke, ae, be), (kh, ah, bh) = self.e, self.h
        dx, ch = cfg.dx, cfg.dt / cfg.dx / MU0
        by, bx = self.box
        for _ in range(count):
            n = self.n
            dEx, dEy = ez[:, :-1, 1:] - ez[:, :-1, :-1], ez[:, 1:, :-1] - ez[:, :-1, :-1]
            self.phx.mul_(bh).addcmul_(dEx, ah)
            self.phy.mul_(bh[:, None]).addcmul_(dEy, ah[:, None])
            hy.add_(dEx.mul_(kh).add_(self.phx, alpha=dx), alpha=ch)
            hx.sub_(dEy.mul_(kh[:, None]).add_(self.phy, alpha=dx), alpha=ch)
            dHy, dHx = hy[:, 1:, 1:] - hy[:, 1:, :-1], hx[:, 1:, 1:] - hx[:, :-1, 1:]
            self.pex.mul_(be).addcmul_(dHy, ae)
            self.pey.mul_(be[:, None]).addcmul_(dHx, ae[:, None])
            old = ez[:, 1:-1, 1:-1]
            old_box = old[:, by, bx].clone()
            if self.ref:
                # kappa divides both curl terms; rows in the y strips are formed from scratch, without the x term
                curl = dHy - dHx
                cx = (curl * ke).add_(self.pex, alpha=dx)
                cy = (curl * ke[:, None]).sub_(self.pey, alpha=dx)
                curl = torch.where(self.strip[:, None], cy, cx)
            else:
                curl = dHy.mul_(ke).add_(self.pex, alpha=dx).sub_(dHx.mul_(ke[:, None]).add_(self.pey, alpha=dx))
            new = (self.ca * old).addcmul_(self.cb, curl)
            nb = new[:, by, bx]
            nb.sub_(self.cj * self.jp)
            if self.ref:
                f1 = torch.exp(-(((n + 0.5) * cfg.dt + self.delay) / cfg.pulse_tau) ** 2)
                f0 = torch.exp(-(((n - 0.5) * cfg.dt + self.delay) / cfg.pulse_tau) ** 2)
                nb.add_(self.ceic * f1 + self.ceip * f0)
                self.jp.mul_(self.kp).add_(self.bp * (nb - old_box + f1 - f0))
            else:
                new[self.every, self.sy - 1, self.sx - 1] += self._source(n)
                self.jp.mul_(self.kp).add_(self.bp * (nb - old_box))
            old.copy_(new)
            flat = [a.reshape(self.B, -1) for a in (ez, hx, hy)]
            h = torch.where(self.yface, flat[1][:, self.at_h], flat[2][:, self.at_h])
            self.samples.append((h, (flat[0][:, self.at_0] + flat[0][:, self.at_1]) * 0.5))
            self.n += 1
            if len(self.samples) == 256:
                self._fold()
        self._fold()

    def _fold(self):
        if not self.samples:
            return
        k = len(self.samples)
        tJ, tM = (0.0, 0.5) if self.ref else (0.5, 1.0)
        step = np.arange(self.n - k, self.n, dtype=np.float64)
        w = 2 * math.pi * self.freq * self.cfg.dt
        for acc, t0, i in ((self.J, tJ, 0), (self.M, tM, 1)):
            ph = torch.as_tensor(np.exp(-1j * w[:, None] * (step + t0)[None, :]), device=self.dev)
            acc += torch.einsum("fk,kbp->bfp", ph, torch.stack([s[i] for s in self.samples]).to(torch.complex128)) * self.sgn
        self.samples = []

    def _norm(self):
        cfg = self.cfg
        if self.ref:
            w, tau = 2 * math.pi * self.freq, cfg.pulse_tau
            prad = 0.5 / ETA0 * (tau * math.sqrt(math.pi) * np.exp(-(tau * w) ** 2 / 4)) ** 2
            return 1 / (8 * math.pi * ETA0 * prad * cfg.ff_norm)
        n = np.arange(cfg.steps)
        u = ((n + 1) * cfg.dt - cfg.pulse_t0) / cfg.pulse_tau
        s = -u * np.exp(-u * u) * cfg.dt
        S = np.array([np.sum(s * np.exp(-2j * math.pi * f * (n + 1) * cfg.dt)) for f in self.freq])
        return 1 / (8 * math.pi * ETA0 * np.abs(S) ** 2)

    def far(self):
        """D and sqrt(D) e^{jP} as [simulation][freq][angle]."""
        cfg = self.cfg
        yf = np.isin(self.leg, (0, 2))
        fx, fy = self.x + 0.5 * ~yf, self.y + 0.5 * yf
        px, py = (cfg.dx * (v - n / 2 + (1 if self.ref else 0)) for v, n in ((fx, cfg.nx), (fy, cfg.ny)))
        phi = 2 * math.pi * np.arange(cfg.n_angles) / cfg.n_angles
        inv, out = self._norm(), []
        yft = self.yface.to(torch.complex128)
        for i, f in enumerate(self.freq):
            k = 2 * math.pi * f / C0
            W = torch.as_tensor(np.exp(1j * k * (px[:, None] * np.cos(phi) + py[:, None] * np.sin(phi))), device=self.dev)
            N = -(self.J[:, i] * cfg.dx) @ W
            Ly, Lx = (self.M[:, i] * cfg.dx * yft) @ W, (self.M[:, i] * cfg.dx * (1 - yft)) @ W
            c, s = (torch.as_tensor(v, device=self.dev) for v in (np.cos(phi), np.sin(phi)))
            E = -s * Ly + c * Lx + ETA0 * N
            out.append(k * math.sqrt(inv[i]) * E)
        far = torch.stack(out, 1).cpu().numpy()
        return np.abs(far) ** 2, far


def _exact_seconds(cfg, sims):
    each = sims * float(cfg.nx) * cfg.ny * 8 * 3 / 3e12
    return cfg.steps * 46 * max(9e-6, each)


def _fitness(cfg, D, target):
    d = (D.reshape(-1) - np.asarray(target, np.float64).reshape(-1)) ** 2
    if cfg.flags & t.FLAG_REL_FITNESS:
        d = d / np.asarray(target, np.float64).reshape(-1) ** 2
    return -float(d.sum()) / (cfg.n_exc * cfg.n_freq)


def exact(case, seed):
    if case["kind"] == "requests":
        reqs = _requests(case, seed)
        if sum(_exact_seconds(c, 2 * c.n_exc) for c, _ in reqs) > 15:
            return None
        fit = []
        for cfg, v in reqs:
            s = _Exact(cfg, [v, _target_vector(cfg)], range(cfg.n_exc))
            s.step(cfg.steps)
            D = s.far()[0]
            fit.append(_fitness(cfg, D[:cfg.n_exc], D[cfg.n_exc:]))
        return {"fitness": np.array(fit)}
    cfg, vectors = _config(case), list(_vectors(case, seed))
    if case["kind"] == "steps":
        s, frames = _Exact(cfg, vectors, [1]), []
        for _ in range(4):
            s.step(cfg.steps // 4)
            jp = torch.zeros_like(s.ez)
            jp[:, 1:-1, 1:-1][:, s.box[0], s.box[1]] = s.jp
            frames.append(tuple(a[0].cpu().numpy().copy() for a in (s.ez, s.hx, s.hy, jp)))
        far = s.far()[1]
        return {"frames": frames, "J": s.J[0].cpu().numpy(), "M": s.M[0].cpu().numpy(),
                "far": far[0]}
    if case["physics"] == "antenna":
        vectors.append(_target_vector(cfg))
    if _exact_seconds(cfg, len(vectors) * cfg.n_exc) > 18:
        return None
    s = _Exact(cfg, vectors, range(cfg.n_exc))
    s.step(cfg.steps)
    D, far = s.far()
    D = D.reshape(len(vectors), -1)
    if case["physics"] == "antenna":
        target, D = D[-1], D[:-1]
    else:
        target = _measurement(case, cfg)
    fit = np.array([_fitness(cfg, d, target) for d in D])
    if case["kind"] == "batch":
        return {"fitness": fit, "D": D}
    if case["kind"] == "objective":
        return {"fitness": float(fit[0])}
    return {"fitness": float(fit[0]), "far": far.reshape(len(vectors), -1)[0]}
