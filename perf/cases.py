"""The work this framework is asked to do, as cases that can be timed and checked.

A case is a dict of plain values. ``prepare`` builds what a user's program holds
before the call (problems as numpy arrays, for a plan that is being watched the
plan itself), ``run`` makes one pass through the public entry points and returns
what the user reads back, ``exact`` gives the same outputs in 64 bits from plain
torch. Three kinds:

* ``run``: one grid from its problem to its results. A plan holds one problem
  and steps it once through, so a new grid means a new plan: the pass creates
  it, steps it, and reads the traces and the final Ez.
* ``watch``: a plan kept by the program and stepped a few steps at a time, Ez
  read after each (a live view, a snapshot cadence): short calls one by one.
* ``pool``: several shots advanced together by one pool, the traces read when
  all are done (a batch, or the frequencies of a served sweep).
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

import fdtd2d_amd as F

C0 = 2.99792458e8
MU0 = 4e-7 * math.pi
EPS0 = 1.0 / (MU0 * C0 * C0)
CJ = 2.81794e-8  # e^2 / m_e
WATCH_LEAD = 256  # steps behind a watched plan when the program takes it up
WATCH_MOST = 1 << 20  # steps a watched plan can go on for


def listed():
    return [
        # a live view of a small grid: 16 steps a frame, Ez read each time
        _watch("watch_256x192", nx=256, ny=192, npml=12, steps=16, medium="density"),
        # the plain method's own workload: 400 x 400, one source, a linear ramp of plasma
        _run("run_400", nx=400, ny=400, npml=12, steps=2000, medium="density", nsrc=1, profile="linear", fluct=0.0),
        # the reference's Settings.ini: 500 x 3000 material ids, 21 RC lines and the processing line captured
        _run("run_table_500x3000", nx=500, ny=3000, npml=10, steps=1500, medium="table", nsrc=16, rc=21, line=420),
        # an odd, ragged grid of ordinary size with a fluctuating plasma
        _run("run_611x1237", nx=611, ny=1237, npml=10, steps=2000, medium="density", nsrc=8),
        # the small shot of the mixed stream: 1024 x 1024, 4000 steps, run by itself
        _run("run_1024", nx=1024, ny=1024, npml=12, steps=4000, medium="density", nsrc=8),
        # the largest grid of the batch and of the sweeps, by itself
        _run("run_2048", nx=2048, ny=2048, npml=12, steps=2000, medium="density", nsrc=8),
        # the large single grid: 8192 x 8192, 16-element array, 64 detectors
        _run("run_8192", nx=8192, ny=8192, npml=16, steps=4000, medium="density", nsrc=16, ndet=64, fluct=0.02),
        # the uneven batch: sides from 256 to 2048 in steps of 128
        _pool("batch_64", shots=64, low=256, high=2048, side=128, steps=1000, medium="density"),
        # one served request: 16 frequencies over one profile on 896 x 896
        _pool("sweep_16", shots=16, low=896, high=896, side=128, steps=1500, medium="density"),
        # a handful of small odd-sized shots with material tables, their final Ez kept
        _pool("pool_table_8", shots=8, low=150, high=420, side=1, steps=600, medium="table", fields=True),
    ]


def draw(rng: random.Random):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["watch", "run", "run", "run", "pool", "pool"])
    medium = rng.choice(["density", "density", "table"])
    npml = rng.choice([8, 10, 12, 16])
    if kind == "watch":
        return _watch(None, nx=log(96, 700), ny=log(96, 700), npml=npml, steps=log(1, 64), medium=medium)
    if kind == "run":
        nx, ny = log(160, 4096), log(160, 4096)
        steps = min(log(200, 4000), int(3e10 / (nx * ny)))
        few = medium == "table" and rng.random() < 0.5
        return _run(None, nx=nx, ny=ny, npml=npml, steps=steps, medium=medium, nsrc=rng.choice([1, 4, 8, 16]),
                    ndet=rng.choice([4, 16]), profile=rng.choice(["linear", "parabolic"]),
                    fluct=rng.choice([0.0, 0.02, 0.05]), rc=rng.randint(1, 21) if few else 0,
                    line=min(nx, 420) // 2 if few else 0)
    low = log(150, 1024)
    high = min(2048, 2 * low)
    shots = log(2, 48)
    steps = min(log(200, 2000), int(4e10 / (shots * high * high)) + 100)
    return _pool(None, shots=shots, low=low, high=high, side=rng.choice([1, 64, 128]), steps=steps, medium=medium,
                 mix=rng.randint(1, 10 ** 6), fields=shots <= 16 and rng.random() < 0.5)


def _named(case, name):
    return case if name is None else {"name": name, **case}


def _run(name, nx, ny, npml, steps, medium, nsrc=1, ndet=4, profile="parabolic", fluct=0.03, rc=0, line=0):
    return _named({"kind": "run", "nx": nx, "ny": ny, "npml": npml, "steps": steps, "medium": medium, "nsrc": nsrc,
                   "ndet": ndet, "profile": profile, "fluct": fluct, "rc": rc, "line": line}, name)


def _watch(name, nx, ny, npml, steps, medium):
    return _named({"kind": "watch", "nx": nx, "ny": ny, "npml": npml, "steps": steps, "medium": medium, "nsrc": 1,
                   "ndet": 4, "profile": "linear", "fluct": 0.0, "rc": 0, "line": 0}, name)


def _pool(name, shots, low, high, side, steps, medium, mix=0, fields=False):
    return _named({"kind": "pool", "shots": shots, "low": low, "high": high, "side": side, "steps": steps,
                   "medium": medium, "mix": mix, "fields": fields}, name)


# ---------------------------------------------------------------- problems
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _smooth_noise(ny, nx, seed):
    """A Gaussian field of about unit variance, correlated over about 20 cells."""
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    coarse = rs.standard_normal((1, 1, ny // 16 + 3, nx // 16 + 3)).astype(np.float32)
    g = torch.nn.functional.interpolate(torch.from_numpy(coarse).to(_device()), size=(ny, nx), mode="bilinear",
                                        align_corners=False)
    return g[0, 0] * 1.4


def _cpml(p, dt, ds):
    """b and c of the E nodes (P of them) and of the H nodes (P - 1), from the outer edge in."""
    out = []
    for n, off in ((p, 1.0), (p - 1, 1.5)):
        depth = np.clip((p - off - np.arange(n)) / (p - 1), 0.0, 1.0)
        sigma = 0.8 * 4 / (math.sqrt(MU0 / EPS0) * ds) * depth ** 3
        alpha = 0.05 * (1.0 - depth)
        b = np.exp(-(sigma + alpha) * dt / EPS0)
        s = sigma + alpha
        c = np.where(s > 0, sigma * (b - 1.0) / np.where(s > 0, s, 1.0), 0.0)
        out.append((b.astype(np.float32), c.astype(np.float32)))
    return out


def _problem(nx, ny, npml, steps, medium, seed, nsrc=1, ndet=4, profile="parabolic", fluct=0.0, rc=0, line=0,
             freq=None, steady=False, plasma_seed=None):
    """A reflectometry problem: an array at the left edge, detectors beside it, plasma to the right."""
    rng = random.Random(seed)
    freq = freq or rng.uniform(8e9, 40e9)
    grid_freq = 40e9 if plasma_seed is not None else freq  # a sweep keeps one grid for its frequencies
    ds = C0 / grid_freq / 20.0
    crit = EPS0 * (2 * math.pi * (10e9 if plasma_seed is not None else freq)) ** 2 / CJ
    peak = random.Random(plasma_seed if plasma_seed is not None else seed + 1).uniform(0.8, 2.5) * crit
    wp2 = peak * (1 + 6 * fluct) * CJ / EPS0
    dt = 0.99 / math.sqrt(2 * C0 * C0 / (ds * ds) + wp2 / 4)
    i = np.arange(nx)
    x0, x1 = 0.3 * nx, 0.75 * nx
    if profile == "linear":
        prof = np.clip((i - x0) / (0.95 * nx - x0), 0.0, 1.0) * peak
    else:
        prof = np.clip(1.0 - ((i - x1) / (x1 - x0)) ** 2, 0.0, None) * peak
    dens = torch.from_numpy(prof).to(_device()).float()[None, :].expand(ny, nx)
    if fluct > 0 or medium == "table":
        s = plasma_seed if plasma_seed is not None else seed
        dens = dens * (1.0 + max(fluct, 0.02 if medium == "table" else 0.0) * _smooth_noise(ny, nx, s + 7))
    dens = torch.clamp(dens, min=0.0)
    nu = 1e9
    p = dict(nx=nx, ny=ny, npml=npml, nsteps=steps, dt=dt, dx=ds, dy=ds, db=float(np.float32(dt / MU0)), cj=CJ,
             dx_f=float(np.float32(ds)), dy_f=float(np.float32(ds)))
    if medium == "density":
        p.update(medium_kind=F.MEDIUM_DENSITY, density=np.ascontiguousarray(dens.cpu().numpy()), ca0=1.0,
                 cb0=float(np.float32(dt / EPS0)), jz_decay=float(np.float32((1 - nu * dt / 2) / (1 + nu * dt / 2))),
                 jz_dt=dt / (1 + nu * dt / 2))
    else:
        # id 0 vacuum, 1 PEC, 2-3 lossy dielectrics, then plasma ids in 48 levels of density
        levels = 48
        eps = np.full(4 + levels, EPS0)
        sig = np.zeros(4 + levels)
        eps[2], eps[3], sig[2], sig[3] = 2.1 * EPS0, 4.5 * EPS0, 0.001, 0.01
        top = peak * (1 + 6 * max(fluct, 0.02))
        q = torch.clamp((dens / top * levels).floor(), 0, levels - 1).int()
        mat = torch.where(dens > 0.01 * peak, q + 4, torch.zeros_like(q)).cpu().numpy()
        wall = max(2, nx // 60)
        h, g = ny // 5, max(4, nx // 30)
        for j0 in (npml + 4, ny - npml - 4 - h):  # two plates of metal beside the array, dielectric behind them
            mat[j0:j0 + h, npml + 6 + g:npml + 6 + g + wall] = 1
            mat[j0:j0 + h, npml + 6 + g + wall:npml + 6 + 2 * g + wall] = rng.choice([2, 3])
        k = sig * dt / (2 * eps)
        ne = np.zeros(4 + levels)
        ne[4:] = (np.arange(levels) + 0.5) / levels * top
        p.update(medium_kind=F.MEDIUM_TABLE, material=np.ascontiguousarray(mat, np.int32),
                 ca=((1 - k) / (1 + k)).astype(np.float32), cb=((dt / eps) / (1 + k)).astype(np.float32),
                 ne=ne.astype(np.float32), pec_material=1, jz_decay=1.0, jz_dt=dt)
    if npml > 0:
        (be, ce), (bh, ch) = _cpml(npml, dt, ds)
        for ax in ("x", "y"):
            p.update({f"be_{ax}": [be, be], f"ce_{ax}": [ce, ce], f"bh_{ax}": [bh, bh], f"ch_{ax}": [ch, ch]})
    den = np.float32(1.0 / ds)
    p.update(den_ex=np.full(nx - 1, den), den_hx=np.full(nx - 1, den), den_ey=np.full(ny - 1, den),
             den_hy=np.full(ny - 1, den))
    col = npml + 8
    span = ny - 2 * (npml + 3)
    pitch = max(1, min(8, span // max(1, nsrc)))
    j = np.clip(ny // 2 - pitch * (nsrc - 1) // 2 + pitch * np.arange(nsrc), npml + 2, ny - npml - 3)
    steer = math.radians(rng.uniform(0.0, 20.0))
    t = np.arange(steps + 1)[:, None] * dt
    if steady:  # a continuous wave, switched on smoothly
        s = np.repeat(np.sin(2 * math.pi * freq * t) * (1 - np.exp(-t * freq / 2)), nsrc, axis=1)
    else:
        u = t - 6.0 / freq - (np.arange(nsrc) * pitch * ds * math.sin(steer) / C0)[None, :]
        s = np.exp(-((u * freq / 2.0) ** 2)) * np.sin(2 * math.pi * freq * u)
    p.update(src_i=np.full(nsrc, col, np.int32), src_j=j.astype(np.int32), src_table=(-s).astype(np.float32))
    dj = np.clip(ny // 2 - ndet + 2 * np.arange(ndet), npml + 2, ny - npml - 3).astype(np.int32)
    p.update(det_i=np.full(ndet, col + 2, np.int32), det_j=dj, comp_i=np.full(1, col + 2, np.int32),
             comp_j=dj[:1].copy())
    if rc:
        a = np.linspace(0.35 * nx, 0.7 * nx, rc).astype(np.int32)
        p.update(rc_imax=a, rc_i=np.minimum(a + 1, nx - 1).astype(np.int32), rc_jcut=npml + 2, rc_level=0.1,
                 rc_edge0=1e-4)
    if line:
        p.update(line_size=line, line_i0=min(npml + 2, nx - line), line_j=ny // 2, line_begin=steps // 3,
                 line_end=steps)
    return p


def _mix(case):
    """The grid sizes of a pool's shots."""
    rng, n = random.Random(case["mix"]), case["side"]
    most = (case["high"] - case["low"]) // n
    return [tuple(case["low"] + n * rng.randint(0, most) for _ in range(2)) for _ in range(case["shots"])]


def _shots(case, seed):
    """The problems of a pool: frequencies and plasmas by the seed; shots of one size share one profile."""
    rng = random.Random(seed * 7919 + 13)
    out = []
    sweep = case["low"] == case["high"]
    for k, (nx, ny) in enumerate(_mix(case)):
        out.append(_problem(nx, ny, 12, case["steps"], case["medium"], seed * 1009 + k, nsrc=rng.randint(1, 16),
                            profile=rng.choice(["linear", "parabolic"]) if not sweep else "parabolic",
                            fluct=rng.uniform(0.0, 0.05) if not sweep else 0.0,
                            freq=rng.uniform(10e9, 40e9), plasma_seed=seed if sweep else None))
    return out


def _one(case, seed):
    watch = case["kind"] == "watch"
    return _problem(case["nx"], case["ny"], case["npml"], WATCH_MOST if watch else case["steps"], case["medium"],
                    seed * 1009, nsrc=case["nsrc"], ndet=case["ndet"], profile=case["profile"], fluct=case["fluct"],
                    rc=case["rc"], line=case["line"], steady=watch)


# ---------------------------------------------------------------- the passes
def prepare(case, seed):
    if case["kind"] == "pool":
        return {"kind": "pool", "problems": [F.Problem(**p) for p in _shots(case, seed)], "fields": case["fields"]}
    problem = F.Problem(**_one(case, seed))
    if case["kind"] == "run":
        return {"kind": "run", "problem": problem, "steps": case["steps"], "rc": case["rc"], "line": case["line"]}
    plan = F.Plan(problem)
    plan.run(WATCH_LEAD)
    plan.sync()
    return {"kind": "watch", "plan": plan, "steps": case["steps"]}


def run(state):
    if state["kind"] == "watch":
        state["plan"].run(state["steps"])
        return {"ez": state["plan"].read_field(F.EZ)}
    if state["kind"] == "run":
        with F.Plan(state["problem"]) as plan:
            plan.run(state["steps"])
            det, comp = plan.read_detectors()
            out = {"det": det, "comp": comp, "ez": plan.read_field(F.EZ)}
            if state["rc"]:
                out["rc"] = plan.read_rc()
            if state["line"]:
                out["line"] = plan.read_line()
        return out
    with F.Pool() as pool:
        ids = [pool.add(p) for p in state["problems"]]
        while pool.info("running") > 0:
            pool.step(8)
        got = [pool.read_detectors(i) for i in ids]
        ez = [pool.read_field(i, F.EZ) for i in ids] if state["fields"] else []
    return {"det": np.stack([d for d, _ in got]), "comp": np.stack([c for _, c in got]), "ez": ez}


def _sizes(case):
    """(nx, ny, steps, sources, detectors) of each grid of a case."""
    if case["kind"] != "pool":
        return [(case["nx"], case["ny"], case["steps"], case["nsrc"], case["ndet"])]
    return [(nx, ny, case["steps"], 8, 4) for nx, ny in _mix(case)]


def work(case):
    """Medium and source table in, traces and Ez out, once each; 16 operations for a cell and step without plasma
    (H 8, E 8) and 9 more where there is plasma, taken as 60 in 100 cells."""
    by, fl = 0.0, 0.0
    for nx, ny, steps, nsrc, ndet in _sizes(case):
        fl += (16 + 0.6 * 9) * nx * ny * steps
        by += 4.0 * steps * (nsrc + ndet + 3) + (4.0 * nx * ny if case.get("fields", True) else 0.0)
        by += 4.0 * nx * ny + (4.0 * case.get("line", 0) * steps * 2 / 3)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    cost = sum(s * (45 * 8e-6 + nx * ny * 45 * 16 / 2e12) for nx, ny, s, _, _ in _sizes(case))
    if cost > 20:
        return None
    if case["kind"] == "pool":
        got = [_step64(p, case["steps"]) for p in _shots(case, seed)]
        out = {k: np.stack([g[k] for g in got]) for k in ("det", "comp")}
        return {**out, "ez": [g["ez"] for g in got] if case["fields"] else []}
    lead = WATCH_LEAD if case["kind"] == "watch" else 0
    out = _step64(_one(case, seed), case["steps"] + lead)
    if lead:
        return {"ez": out["ez"]}
    if case["rc"]:
        out["rc"] = None
    if not case["line"]:
        out.pop("line")
    return out


def _step64(p, steps):
    """The update equations on whole planes in float64 (psi carried on the whole grid, zero outside the strips)."""
    dev = torch.device(_device())
    f8 = torch.float64

    def t(a):
        return torch.as_tensor(np.asarray(a, np.float64), dtype=f8, device=dev)

    nx, ny, n = p["nx"], p["ny"], p["npml"]
    ez, hx, hy, jz = (torch.zeros((ny, nx), dtype=f8, device=dev) for _ in range(4))
    db, cj, jdt, decay = p["db"], float(np.float32(p["cj"])), p["jz_dt"], p["jz_decay"]
    if p["medium_kind"] == F.MEDIUM_TABLE:
        m = torch.as_tensor(p["material"], device=dev).long()
        ca, cb, ne, pec = t(p["ca"])[m], t(p["cb"])[m], t(p["ne"])[m], m == p["pec_material"]
    else:
        ca, cb, ne, pec = p["ca0"], p["cb0"], t(p["density"]), None
    inner = (slice(1, ny - 1), slice(1, nx - 1))
    drive = cj * jdt * ne[inner]
    keep = torch.where(ne[inner] > 0, decay, 1.0).to(f8)
    if pec is not None:
        ca, cb, pec = ca[inner], cb[inner], pec[inner]
    # b and c of every row / column of the H updates (rows 0..n-2) and the E updates (1..n-2)
    tables = {}
    for ax, size in (("x", nx), ("y", ny)):
        h = np.zeros((2, size - 1))
        e = np.zeros((2, size - 2))
        for r in range(n - 1 if n else 0):
            h[:, r] = p[f"bh_{ax}"][0][r], p[f"ch_{ax}"][0][r]
            h[:, size - 2 - r] = p[f"bh_{ax}"][1][r], p[f"ch_{ax}"][1][r]
        for r in range(1, n):
            e[:, r - 1] = p[f"be_{ax}"][0][r], p[f"ce_{ax}"][0][r]
            e[:, size - 2 - r] = p[f"be_{ax}"][1][r], p[f"ce_{ax}"][1][r]
        d = p[f"d{ax}_f"]
        shape = (1, -1) if ax == "x" else (-1, 1)
        tables[ax] = [t(v).reshape(shape) for v in (h[0], h[1] / d, e[0], e[1] / d)]
    bhx, chx, bex, cex = tables["x"]
    bhy, chy, bey, cey = tables["y"]
    hxy, hyx = (torch.zeros((ny - 1, nx - 1), dtype=f8, device=dev) for _ in range(2))
    ezx, ezy = (torch.zeros((ny - 2, nx - 2), dtype=f8, device=dev) for _ in range(2))
    den_hy, den_hx = t(p["den_hy"])[:, None], t(p["den_hx"])[None, :]
    den_ey, den_ex = t(p["den_ey"])[1:, None], t(p["den_ex"])[None, 1:]
    src = t(p["src_table"][: steps + 1])
    idx = {k: torch.as_tensor(p[k].astype(np.int64), device=dev)
           for k in ("src_i", "src_j", "det_i", "det_j", "comp_i", "comp_j")}
    traced = p["nsteps"] < WATCH_MOST  # a watched plan's traces are not read
    det = torch.zeros((p["nsteps"] + 1 if traced else 1, len(p["det_i"])), dtype=f8, device=dev)
    comp = torch.zeros((3, det.shape[0], len(p["comp_i"])), dtype=f8, device=dev)
    size = p.get("line_size", 0)
    rows = max(0, p["line_end"] - p["line_begin"]) if size else 0
    line = torch.zeros((rows, size), dtype=f8, device=dev)
    for s in range(1, steps + 1):
        dy = ez[:-1, :-1] - ez[1:, :-1]
        dx = ez[:-1, 1:] - ez[:-1, :-1]
        hxy.mul_(bhy).add_(chy * dy)
        hyx.mul_(bhx).add_(chx * dx)
        hx[:-1, :-1] += db * (dy * den_hy + hxy)
        hy[:-1, :-1] += db * (dx * den_hx + hyx)
        dhy = hy[1:-1, 1:-1] - hy[1:-1, :-2]
        dhx = hx[:-2, 1:-1] - hx[1:-1, 1:-1]
        ezx.mul_(bex).add_(cex * dhy)
        ezy.mul_(bey).add_(cey * dhx)
        e = ez[inner]
        jz[inner] = jz[inner] * keep + drive * e
        main = ca * e + cb * (dhy * den_ex + dhx * den_ey - jz[inner])
        if pec is not None:
            main = torch.where(pec, torch.zeros_like(main), main)
        ez[inner] = main + cb * (ezx + ezy)
        ez.index_put_((idx["src_j"], idx["src_i"]), -src[s], accumulate=True)
        if traced:
            det[s] = ez[idx["det_j"], idx["det_i"]]
            for q, f in enumerate((ez, hx, hy)):
                comp[q, s] = f[idx["comp_j"], idx["comp_i"]]
        if rows and p["line_begin"] < s <= p["line_end"]:
            line[s - p["line_begin"] - 1] = ez[p["line_j"], p["line_i0"]:p["line_i0"] + size]
    return {k: v.cpu().numpy() for k, v in (("det", det), ("comp", comp), ("ez", ez), ("line", line))}
