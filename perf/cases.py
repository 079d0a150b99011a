"""The work users of this package give it, as measurable cases.

Kinds of case (`case["kind"]`):
  steps      pseudo-time steps of one grid (Solver.iterate), then the new state read back
  tasks      the same steps as separate task calls, the way OneFLOW's task list drives the library
  residual   back-to-back NS + SA residual evaluations of one state, then the residual read back
  zones      several airfoil cases advanced as zones of one context
  train      training steps of the warm-start network
  gradients  its loss and the gradient of every parameter on one batch
  forward    its forward pass on host samples
  serve      its allocation-free forward pass on device samples

Grids come from the package's generators and from the reference grids its
tests hold; flow conditions, starting fields, network weights and samples
from the seed.
"""
import ctypes
import functools
import math
from pathlib import Path

import numpy as np
import torch

from oneflow_amd import meshgen
from oneflow_amd.cases import airfoil_sweep
from oneflow_amd.config import CaseConfig
from oneflow_amd.mesh import read_ofl
from oneflow_amd.mlp import Mlp
from oneflow_amd.solver import Solver, ZoneSolver

ROOT = Path(__file__).resolve().parent.parent
LAYERS = [(16, 256)] + 4 * [(256, 256)] + [(256, 64)]  # padded network shapes (9 inputs, 5 outputs used)


def listed():
    return [
        # A small laminar plate in structured numbering, every step's norms read (res.dat rows): a
        # regression test or a first run, all latency and launches.
        dict(name="plate_small", kind="steps", grid="plate", a=41, b=25, order="natural", scheme="slau2", ilim=0,
             visc="laminar", steps=50, norms=True),
        # The reference's RAE2822 case on its own grid and numbering (23,552 cells), as its users run it.
        dict(name="rae2822", kind="steps", grid="rae2822_roe_sa", order="natural", scheme="roe", ilim=2, visc="sa",
             steps=20, norms=True),
        # The benchmark's NACA0012 (120,832 cells) in the generator's structured numbering.
        dict(name="naca_natural", kind="steps", grid="naca", a=512, b=98, order="natural", scheme="roe", ilim=2,
             visc="sa", steps=20, norms=False),
        # The same grid coloured, the numbering the package recommends: a production 2-D run.
        dict(name="naca_coloured", kind="steps", grid="naca", a=512, b=98, order="colour", scheme="roe", ilim=2,
             visc="sa", steps=200, norms=False),
        # The drop-in's task calls on a mid-size airfoil with norms each step (the host keeps the step loop).
        dict(name="tasks", kind="tasks", grid="naca", a=256, b=70, order="colour", scheme="roe", ilim=2, visc="sa",
             steps=40, norms=True),
        # The benchmark's residual evaluation on the NACA0012 grid.
        dict(name="naca_residual", kind="residual", grid="naca", a=512, b=98, order="colour", scheme="roe", ilim=2,
             visc="sa", evals=200),
        # The benchmark's 3-D swept wing (2,524,160 prisms and tets), the largest single-GPU run.
        dict(name="wing_steps", kind="steps", grid="wing", a=34, b=0, order="colour", scheme="roe", ilim=2, visc="sa",
             steps=60, norms=False),
        # The same wing, fewer span layers: residual evaluations of the FP32-flux variant.
        dict(name="wing_fp32", kind="residual", grid="wing", a=8, b=0, order="colour", scheme="roe", ilim=2, visc="sa",
             evals=100, fp32=True),
        # A sweep of uneven airfoil grids as zones, first order, as the warm-start experiment solves them.
        dict(name="zones", kind="zones", n=16, sweep=2026, low=20000, high=60000, ilim=-1, steps=50),
        # Training the warm-start network with its default batch.
        dict(name="mlp_train", kind="train", samples=65536, batch=8192, steps=60),
        # Its prediction of a whole sweep's start field, from host memory.
        dict(name="mlp_forward", kind="forward", n=1_000_003),
        # Its allocation-free forward on a few device-resident samples (a serving loop, 100 calls).
        dict(name="mlp_serve", kind="serve", n=500, calls=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "steps", "tasks", "residual", "zones", "train", "gradients",
                       "forward", "serve"])
    if kind == "zones":
        n = _log(rng, 2, 12)
        return dict(kind=kind, n=n, sweep=rng.randrange(1 << 20), low=20000, high=_log(rng, 24000, 90000),
                    ilim=rng.choice([-1, 2]), steps=_log(rng, 10, 50))
    if kind == "train":
        return dict(kind=kind, samples=_log(rng, 3000, 100000), batch=_log(rng, 200, 10000), steps=_log(rng, 10, 60))
    if kind == "gradients":
        return dict(kind=kind, n=_log(rng, 60, 30000))
    if kind == "forward":
        return dict(kind=kind, n=_log(rng, 1, 1_100_000))
    if kind == "serve":
        return dict(kind=kind, n=_log(rng, 1, 8192), calls=100)
    grid = rng.choice(["plate", "naca", "naca", "wing"])
    c = dict(kind=kind, grid=grid, order=rng.choice(["natural", "colour"]))
    if grid == "plate":
        c.update(a=_log(rng, 31, 241), b=_log(rng, 17, 129))
        c.update(scheme=rng.choice(["roe", "slau2"]), ilim=rng.choice([-1, 0, 2]), visc=rng.choice(["euler", "laminar"]))
    elif grid == "naca":
        c.update(a=8 * _log(rng, 12, 76), b=_log(rng, 24, 120))
        c.update(scheme=rng.choice(["roe", "slau2"]), ilim=rng.choice([-1, 1, 2]), visc="sa")
    else:
        c.update(a=rng.randint(2, 12), b=0, scheme="roe", ilim=rng.choice([-1, 2]), visc="sa")
    if kind == "residual":
        c.update(evals=_log(rng, 20, 100), fp32=rng.random() < 0.3)
    else:
        c.update(steps=_log(rng, 10, 60), norms=rng.random() < 0.5)
        if kind == "steps" and rng.random() < 0.15:
            c.update(rk=rng.randint(1, 3), ilim=-1)  # explicit multi-stage steps
    return c


# ---------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=None)
def _grid(grid, a, b, order):
    if grid == "plate":
        g = meshgen.flat_plate(a, b)
    elif grid == "naca":
        g = meshgen.naca_hybrid(n_surf=a, n_quad=40, ratio=1.15, reynolds=6.5e6, n_outer=b, radius=30.0)
    elif grid == "wing":
        g = meshgen.swept_wing(n_span=a)
    else:
        g = read_ofl(ROOT / "tests" / "golden" / "reference" / grid / "grid.ofl")
    if order == "colour":
        o = meshgen.multicolor_order(g)
        g = meshgen.renumber(g, o)
        if grid == "wing":  # large 3-D grids keep their interior faces in spatial order
            g = meshgen.sort_interior_faces(g, o)
    return g


@functools.lru_cache(maxsize=4)
def _sweep(n, seed, low, high):
    cases = airfoil_sweep(n, seed=seed, min_cells=low, max_cells=high)
    return [c.grid("multicolor") for c in cases], [c.reynolds for c in cases]


def _case_grid(case):
    return _grid(case["grid"], case.get("a", 0), case.get("b", 0), case["order"])


def _config(case, rng):
    """The run's script keys; Mach, incidence and Reynolds number from the seed."""
    if case["grid"] == "plate":
        flow = dict(mach_ref=rng.uniform(0.1, 0.3), reynolds=rng.uniform(2e5, 5e6))
    elif case["grid"] == "wing":
        flow = dict(mach_ref=rng.uniform(0.75, 0.84), aoa_degree=rng.uniform(1.0, 3.0), reynolds=rng.uniform(1e7, 1.2e7))
    else:
        flow = dict(mach_ref=rng.uniform(0.5, 0.8), aoa_degree=rng.uniform(0.0, 2.5), reynolds=rng.uniform(6e6, 7e6))
    rk = case.get("rk", 0)
    return CaseConfig(dim=3 if case["grid"] == "wing" else 2, ischeme=1 if case["scheme"] == "roe" else 12,
                      ilim=case["ilim"], vismodel={"euler": 0, "laminar": 1, "sa": 3}[case["visc"]], centropy1=0.001,
                      centropy2=0.001, vencat_coef=0.001, flux_fp32=int(case.get("fp32", False)),
                      time_integral=1 if rk else 2, rk_stage=max(rk, 1), **(dict(cflst=0.1, cfled=0.2) if rk else {}),
                      **flow)


def _freestream(cfg):
    a = math.radians(cfg.aoa_degree)
    return [1.0, math.cos(a), math.sin(a), 0.0, 1.0 / (cfg.gama_ref * cfg.mach_ref ** 2)]


def _field(g, cfg, rng):
    """A smooth state around freestream with cell-scale noise: [5][cells] and nu_tilde [cells]."""
    xyz = meshgen.cell_centroids(g)
    w = [0.02 * np.sin(xyz @ rng.normal(0.0, 2.0, 3) + rng.uniform(0, 6.3)) + 0.002 * rng.standard_normal(g.n_cells)
         for _ in range(5)]
    q = np.zeros((5, g.n_cells))
    free = _freestream(cfg)
    for e in range(5):
        q[e] = free[e] * (1.0 + w[e]) if e in (0, 4) else free[e] + w[e]
    if g.dim == 2:
        q[3] = 0.0
    return q, cfg.ref_sa * (1.0 + 5.0 * np.abs(w[3]))


def _set_state(s, q, nu):
    full = s.get("Q")
    full[:, :q.shape[1]] = q
    s.set("Q", full)
    t = s.get("TURBQ")
    t[:nu.shape[0]] = nu
    s.set("TURBQ", t)
    s.ns_boundary()
    s.sa_boundary()


def _params(rng):
    """Network parameters in the library's layout: per layer W[kin][kout], then b[kout]."""
    out = []
    for k, (ki, ko) in enumerate(LAYERS):
        ni, no = (9 if k == 0 else ki), (5 if k == 5 else ko)
        w, b = np.zeros((ki, ko)), np.zeros(ko)
        w[:ni, :no] = rng.uniform(-1, 1, (ni, no)) * math.sqrt(6.0 / ni)
        b[:no] = 0.1 * rng.standard_normal(no)
        out += [w.ravel(), b]
    return np.concatenate(out).astype(np.float32)


def _samples(rng, n):
    x = rng.standard_normal((n, 9)).astype(np.float32)
    t = np.tanh(x[:, :5] * x[:, 4:9]).astype(np.float32)
    return x, t


@functools.lru_cache(maxsize=None)
def _stream():
    return torch.cuda.Stream()  # the library's fixed work array serves one stream at a time


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("train", "gradients", "forward", "serve"):
        net = Mlp(seed=seed & 0xFFFF)
        net.set_params(_params(rng))
        if kind == "serve":
            x = torch.from_numpy(_samples(rng, case["n"])[0]).cuda()
            return dict(case=case, net=net, x=x, y=torch.zeros(case["n"], 5, device="cuda"), stream=_stream())
        x, t = _samples(rng, case["samples"] if kind == "train" else case["n"])
        return dict(case=case, net=net, x=x, t=t)
    if kind == "zones":
        grids, re = _sweep(case["n"], case["sweep"], case["low"], case["high"])
        cfgs = [CaseConfig(ischeme=1, ilim=case["ilim"], vismodel=3, mach_ref=rng.uniform(0.3, 0.8),
                           aoa_degree=rng.uniform(-2, 6), reynolds=r, centropy1=0.001, centropy2=0.001,
                           vencat_coef=0.001) for r in re]
        s = ZoneSolver(grids, cfgs)
        s.init_freestream()
        s.iterate(1, 20, with_norms=False)
        return dict(case=case, s=s, it=21)
    g, cfg = _case_grid(case), _config(case, rng)
    s = Solver(g, cfg)
    s.init_freestream()
    _set_state(s, *_field(g, cfg, rng))
    if kind == "residual":
        s.timestep(cfg.ncfl)
        s.sync()
        return dict(case=case, s=s)
    s.iterate(1, 10, with_norms=False)
    return dict(case=case, s=s, it=11)


# ---------------------------------------------------------------- one pass

def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "train":
        loss = state["net"].train(state["x"], state["t"], batch=case["batch"], steps=case["steps"])
        return {"losses": loss, "params": state["net"].params()}
    if kind == "gradients":
        loss, grad = state["net"].gradients(state["x"], state["t"])
        return {"loss": loss, "grad": grad}
    if kind == "forward":
        return {"y": state["net"].forward(state["x"])}
    if kind == "serve":
        net, x, y = state["net"], state["x"], state["y"]
        for _ in range(case["calls"]):
            if net._L.ofx_mlp_forward_noalloc(net.h, x.data_ptr(), case["n"], y.data_ptr(),
                                              ctypes.c_void_p(state["stream"].cuda_stream)) != 0:
                raise RuntimeError(net._L.ofx_last_error().decode())
        return {"y": y}
    s = state["s"]
    C = s.n_cells
    if kind == "residual":
        for _ in range(case["evals"]):
            s.residual_ns()
            if case["visc"] == "sa":
                s.residual_sa()
        return {"res": s.get("RES")[:, :C], "turbres": s.get("TURBRES")[:C]}
    n, it = case["steps"], state["it"]
    state["it"] += n
    out = {}
    if kind == "zones":
        s.iterate(it, n, with_norms=False)
        out.update(norms=s.zone_norms(), forces=s.zone_aero())
    elif kind == "tasks":
        sa, norms = case["visc"] == "sa", []
        for k in range(n):
            s.timestep(it + k)
            s.residual_ns()
            s.lusgs_ns()
            s.update_ns()
            s.ns_boundary()
            if sa:
                s.residual_sa()
                s.lusgs_sa()
                s.update_sa()
                s.sa_boundary()
            if case["norms"]:
                norms.append(s.norms())
        if norms:
            out["norms"] = np.array(norms)
    else:
        norms = s.iterate(it, n, with_norms=case["norms"])
        if norms is not None:
            out["norms"] = norms
    out["q"] = s.get("Q")
    if case.get("visc", "sa") == "sa":
        out["nu"] = s.get("TURBQ")
    return out


# ---------------------------------------------------------------- work

def work(case):
    """Each step or evaluation reads the grid's geometry and its state once and writes its result once."""
    kind = case["kind"]
    macs = sum(a * b for a, b in LAYERS[1:-1]) + 9 * 256 + 256 * 5
    params = sum(a * b + b for a, b in LAYERS)
    if kind == "train":
        rows = case["steps"] * min(case["batch"], case["samples"])
        return dict(bytes=4.0 * (14 * rows + 6 * params * case["steps"]), flops=6.0 * macs * rows)
    if kind == "gradients":
        return dict(bytes=4.0 * (14 * case["n"] + 2 * params), flops=6.0 * macs * case["n"])
    if kind in ("forward", "serve"):
        n = case["n"] * case.get("calls", 1)
        return dict(bytes=4.0 * 14 * n + 2.0 * params * case.get("calls", 1), flops=2.0 * macs * n)
    if kind == "zones":
        grids = _sweep(case["n"], case["sweep"], case["low"], case["high"])[0]
    else:
        grids = [_case_grid(case)]
    C, F = sum(g.n_cells for g in grids), sum(g.n_faces for g in grids)
    sa = case.get("visc", "sa") == "sa"
    reps = case.get("steps", case.get("evals"))
    state = 8.0 * (6 if sa else 5) * C
    geom = 64.0 * F + (40.0 if sa else 32.0) * C  # normal, area, centre, two ids; centre, volume, wall distance
    per_face, per_cell = (600, 700) if kind == "residual" else (1100, 1200)
    return dict(bytes=reps * (2 * state + geom), flops=float(reps) * (per_face * F + per_cell * C))


# ---------------------------------------------------------------- 64-bit values

def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("forward", "serve", "gradients"):
        p = _params(rng)
        x, t = _samples(rng, case["n"])
        x, t = torch.from_numpy(x).double(), torch.from_numpy(t).double()
        ws, o = [], 0
        for ki, ko in LAYERS:
            w = torch.from_numpy(p[o:o + ki * ko].reshape(ki, ko)).double()
            b = torch.from_numpy(p[o + ki * ko:o + ki * ko + ko]).double()
            ws += [w.requires_grad_(kind == "gradients"), b.requires_grad_(kind == "gradients")]
            o += ki * ko + ko
        if kind != "gradients":
            return {"y": torch.cat([_network(ws, c) for c in x.split(1 << 16)]).numpy()}
        loss = ((_network(ws, x) - t) ** 2).mean()
        loss.backward()
        return {"loss": float(loss), "grad": torch.cat([w.grad.reshape(-1) for w in ws]).numpy()}
    if kind == "residual" and case["grid"] == "naca" and case["ilim"] == 2 and case["scheme"] == "roe":
        g, cfg = _case_grid(case), _config(case, rng)
        res, turbres = _residual_2d(g, cfg, *_field(g, cfg, rng))
        return {"res": res, "turbres": turbres}
    return None  # long runs of steps, and flows whose wall distance alone takes longer than is useful


def _network(ws, x):
    h = torch.nn.functional.pad(x, (0, 7))
    for k in range(5):
        h = torch.nn.functional.silu(h @ ws[2 * k] + ws[2 * k + 1])
    return (h @ ws[10] + ws[11])[:, :5]


def _residual_2d(g, cfg, q, nu):
    """NS and SA residual of a 2-D airfoil state: Roe with entropy fix, Venkatakrishnan limiter,
    Green-Gauss gradients, standard viscous face gradients, SA with first-order convection."""
    C, B, F = g.n_cells, g.n_bfaces, g.n_faces
    l = g.lc.astype(np.int64)
    r = np.where(np.arange(F) < B, C + np.arange(F), g.rc)
    inner = slice(B, F)
    n1, n2 = g.face_nodes.reshape(-1, 2).T
    dx, dy = g.y[n2] - g.y[n1], g.x[n1] - g.x[n2]
    area = np.hypot(dx, dy)
    nx, ny = dx / area, dy / area
    xf, yf = 0.5 * (g.x[n1] + g.x[n2]), 0.5 * (g.y[n1] + g.y[n2])

    def gather(v):  # sum over each cell's faces, outward sign
        return np.bincount(l, v, C) - np.bincount(r[inner], v[inner], C)
    dot = (xf * nx + yf * ny) * area
    vol = 0.5 * gather(dot)
    xc, yc = gather(xf * dot) / (3.0 * vol), gather(yf * dot) / (3.0 * vol)
    lb = l[:B]
    mir = 2.0 * ((xc[lb] - xf[:B]) * nx[:B] + (yc[lb] - yf[:B]) * ny[:B])
    xc, yc = np.append(xc, xc[lb] - nx[:B] * mir), np.append(yc, yc[lb] - ny[:B] * mir)
    vol = np.append(vol, vol[lb])
    wall = np.flatnonzero(g.bc_type == 2)
    dist = np.full(C, np.inf)
    for f in wall:
        ax, ay, bx, by = g.x[n1[f]], g.y[n1[f]], g.x[n2[f]], g.y[n2[f]]
        ex, ey = bx - ax, by - ay
        t = np.clip(((xc[:C] - ax) * ex + (yc[:C] - ay) * ey) / (ex * ex + ey * ey), 0.0, 1.0)
        dist = np.minimum(dist, (xc[:C] - ax - t * ex) ** 2 + (yc[:C] - ay - t * ey) ** 2)
    dist = np.sqrt(dist)

    gam, gm1 = cfg.gama_ref, cfg.gama_ref - 1.0
    coef, ore = 1.0 / (gam * cfg.mach_ref ** 2), 1.0 / cfg.reynolds
    ts = 110.4 / cfg.tref_dim
    free = np.array(_freestream(cfg))
    is_wall = g.bc_type == 2
    # ghosts: adiabatic wall, characteristic far field
    ro, uo, vo, _, po = q[:, lb]
    fx, fy = nx[:B], ny[:B]
    vin, vref = fx * uo + fy * vo, fx * free[1] + fy * free[2]
    cin, cref = np.sqrt(gam * po / ro), math.sqrt(gam * free[4])
    rp, rm = vin + 2.0 * cin / gm1, vref - 2.0 * cref / gm1
    vnb, cb = 0.5 * (rp + rm), 0.25 * (rp - rm) * gm1
    out = vnb >= 0.0
    entr = np.where(out, po / ro ** gam, free[4])
    ut, vt = np.where(out, uo - fx * vin, free[1] - fx * vref), np.where(out, vo - fy * vin, free[2] - fy * vref)
    rb = (cb * cb / (entr * gam)) ** (1.0 / gm1)
    far = np.array([rb, ut + fx * vnb, vt + fy * vnb, 0.0 * rb, cb * cb * rb / gam])
    sup = np.hypot(uo, vo) > cin
    far = np.where(sup, np.where(vin >= 0.0, q[:, lb], free[:, None]), far)
    nufar = np.where(np.where(sup, vin, vnb) >= 0.0, nu[lb], cfg.ref_sa)
    q = np.concatenate([q, np.where(is_wall, np.array([ro, -uo, -vo, 0.0 * ro, po]), far)], axis=1)
    nu = np.append(nu, np.where(is_wall, -nu[lb], nufar))
    rho, u, v, _, p = q
    T = p / (coef * rho)
    mul = np.sqrt(T ** 3) * (1 + ts) / (T + ts)
    chi = nu[:C] * rho[:C] / mul[:C]
    mut = chi ** 3 / (chi ** 3 + 7.1 ** 3) * rho[:C] * nu[:C]
    mut = np.append(np.minimum(mut, mul[:C] * cfg.max_vis_ratio), np.minimum(mut, mul[:C] * cfg.max_vis_ratio)[lb])

    d1, d2 = np.hypot(xf - xc[l], yf - yc[l]), np.hypot(xf - xc[r], yf - yc[r])
    cl, cr = d2 / (d1 + d2), d1 / (d1 + d2)

    def grad(w):
        face = (cl * w[l] + cr * w[r]) * area
        gx, gy = gather(face * nx) / vol[:C], gather(face * ny) / vol[:C]
        return np.append(gx, gx[lb]), np.append(gy, gy[lb])
    li, ri = l[inner], r[inner]

    def limiter(w, gr):
        mn, mx = w[:C].copy(), w[:C].copy()
        for a, b in ((li, ri), (ri, li)):
            np.minimum.at(mn, a, w[b])
            np.maximum.at(mx, a, w[b])
        mn, mx = mn - w[:C], mx - w[:C]
        eps = (cfg.vencat_coef * max(mx.max() - mn.min(), 1.0)) ** 2
        phi = np.ones(C)
        for c, sel in ((l, slice(0, F)), (ri, inner)):
            y = gr[0][c] * (xf[sel] - xc[c]) + gr[1][c] * (yf[sel] - yc[c])
            x = np.where(y > 0.0, mx[c], mn[c])
            f = np.where(y == 0.0, 1.0, (x * x + eps + 2 * x * y) / (x * x + 2 * y * y + x * y + eps))
            np.minimum.at(phi, c, f)
        return phi
    qs = [rho, u, v, p]
    gr = [grad(w) for w in qs]
    L, R = [], []
    for w, gw in zip(qs, gr):
        ph = limiter(w, gw)
        pf = np.minimum(ph[li], ph[ri])
        a, b = 0.5 * (w[l] + w[r]), 0.5 * (w[l] + w[r])
        a[inner] = w[li] + pf * (gw[0][li] * (xf - xc[l])[inner] + gw[1][li] * (yf - yc[l])[inner])
        b[inner] = w[ri] + pf * (gw[0][ri] * (xf - xc[r])[inner] + gw[1][ri] * (yf - yc[r])[inner])
        L.append(a)
        R.append(b)
    for k in range(4):
        fix = 0.0 * rho[l[wall]] if k in (1, 2) else qs[k][l[wall]]
        L[k][wall], R[k][wall] = fix, fix
    for S, c in ((L, l), (R, r)):
        bad = (S[0] <= 0.0) | (S[3] <= 0.0)
        bad[:B] = False
        for k in range(4):
            S[k] = np.where(bad, qs[k][c], S[k])
    rl, ul, vl, pl = L
    rr, ur, vr, pr = R
    hl, hr = gam / gm1 * pl / rl + 0.5 * (ul ** 2 + vl ** 2), gam / gm1 * pr / rr + 0.5 * (ur ** 2 + vr ** 2)
    vnl, vnr = nx * ul + ny * vl, nx * ur + ny * vr
    s = np.sqrt(rr / rl)
    um, vm, hm = ((a + b * s) / (1.0 + s) for a, b in ((ul, ur), (vl, vr), (hl, hr)))
    v2, vn = um ** 2 + vm ** 2, nx * um + ny * vm
    c2 = gm1 * (hm - 0.5 * v2)
    c = np.sqrt(np.abs(c2))
    e1, e2, e3 = np.abs(vn), np.abs(vn + c), np.abs(vn - c)
    top = np.maximum(e2, e3)
    e1 = np.maximum(top * cfg.centropy1, e1)
    e2, e3 = np.maximum(top * cfg.centropy2, e2), np.maximum(top * cfg.centropy2, e3)
    dq = [rr - rl, rr * ur - rl * ul, rr * vr - rl * vl, rr * hr - pr - (rl * hl - pl)]
    x1, x2 = (2 * e1 - e2 - e3) / (2 * c2), (e2 - e3) / (2 * c)
    dc = vn * dq[0] - nx * dq[1] - ny * dq[2]
    dh = gm1 * (dq[3] - um * dq[1] - vm * dq[2] + 0.5 * v2 * dq[0])
    t1, t2 = dh * x1 + dc * x2, c2 * dc * x1 + dh * x2
    flux = [rl * vnl + rr * vnr - (e1 * dq[0] - t1),
            rl * vnl * ul + rr * vnr * ur + nx * (pl + pr) - (e1 * dq[1] - um * t1 + nx * t2),
            rl * vnl * vl + rr * vnr * vr + ny * (pl + pr) - (e1 * dq[2] - vm * t1 + ny * t2),
            rl * vnl * hl + rr * vnr * hr - (e1 * dq[3] - hm * t1 + vn * t2)]
    # viscous flux: averaged gradients corrected along the centre line
    ex, ey = xc[r] - xc[l], yc[r] - yc[l]
    ol = 1.0 / np.hypot(ex, ey)
    ex, ey = ex * ol, ey * ol

    def face_grad(w, gw):
        gx, gy = 0.5 * (gw[0][l] + gw[0][r]), 0.5 * (gw[1][l] + gw[1][r])
        df = (w[r] - w[l]) * ol - (gx * ex + gy * ey)
        return gx + df * ex, gy + df * ey
    ux, uy = face_grad(u, gr[1])
    vx, vy = face_grad(v, gr[2])
    tx, ty = face_grad(T, grad(T))
    ml, mt = 0.5 * (mul[l] + mul[r]), 0.5 * (mut[l] + mut[r])
    mu = ml + mt
    cp = 1.0 / (gm1 * cfg.mach_ref ** 2)
    div = 2.0 / 3.0 * (ux + vy)
    sx = mu * (nx * (2 * ux - div) + ny * (uy + vx))
    sy = mu * (nx * (uy + vx) + ny * (2 * vy - div))
    heat = (ml / cfg.prl + mt / cfg.prt) * cp * (nx * tx + ny * ty)
    se = 0.5 * (u[l] + u[r]) * sx + 0.5 * (v[l] + v[r]) * sy + heat
    tot = [area * (0.5 * f) - ore * area * s for f, s in zip(flux, (0.0, sx, sy, se))]
    res = np.zeros((5, C))
    for k, e in enumerate((0, 1, 2, 4)):
        res[e] = -gather(tot[k])
    # SA
    gn = grad(nu)
    u1, v1, u2, v2f, na, nb = u[l].copy(), v[l].copy(), u[r].copy(), v[r].copy(), nu[l].copy(), nu[r].copy()
    for a, b in ((u1, u2), (v1, v2f), (na, nb)):
        a[:B] = b[:B] = 0.5 * (a[:B] + b[:B])
    for a in (u1, u2, v1, v2f):
        a[wall] = 0.0
    cn1, cn2 = nx * u1 + ny * v1, nx * u2 + ny * v2f
    conv = area * (np.maximum(cn1, 0.0) * na + np.minimum(cn2, 0.0) * nb)
    ax, ay, bx, by = xc[l] - xf, yc[l] - yf, xc[r] - xf, yc[r] - yf
    s1, s2 = nx * ax + ny * ay, nx * bx + ny * by
    g1 = np.degrees(np.arcsin(np.clip(-s1 / np.hypot(ax, ay), -1, 1)))
    g2 = np.degrees(np.arcsin(np.clip(s2 / np.hypot(bx, by), -1, 1)))
    skew = (g1 > 20.0) & (g2 > 20.0)
    w1 = nu[l] + np.where(skew, gn[0][l] * (nx * s1 - ax) + gn[1][l] * (ny * s1 - ay), 0.0)
    w2 = nu[r] + np.where(skew, gn[0][r] * (nx * s2 - bx) + gn[1][r] * (ny * s2 - by), 0.0)
    mid = 0.5 * (nu[l] + nu[r])
    c1 = s1 * s1 / (s1 * s1 + s2 * s2)
    c1[:B] = 1.0
    dndn = np.where((g1 > 0) & (g2 > 0), c1 * (w1 - mid) / s1 + (1.0 - c1) * (w2 - mid) / s2, 0.0)
    diff = -ore * (0.5 * (mul[l] / rho[l] + mul[r] / rho[r]) + mid) * 1.5 * dndn * area
    k2, cb1, cb2 = 0.41 ** 2, 0.1355, 0.622
    cw1 = cb1 / k2 + (1.0 + cb2) * 1.5
    vort = np.abs(gr[2][0][:C] - gr[1][1][:C])
    nc = nu[:C]
    fv1 = chi ** 3 / (chi ** 3 + 7.1 ** 3)
    fv2 = 1.0 - chi / (1.0 + chi * fv1)
    rs = nc * ore / (k2 * dist ** 2)
    sb = rs * fv2
    st = np.where(sb >= -0.7 * vort, vort + sb, vort + vort * (0.49 * vort + 0.9 * sb) / ((0.9 - 1.4) * vort - sb))
    rr_ = np.minimum(rs / st, 10.0)
    gg = rr_ + 0.3 * (rr_ ** 6 - rr_)
    fw = gg * (65.0 / (gg ** 6 + 64.0)) ** (1.0 / 6.0)
    prod = cb1 * st * nc
    src = prod - cw1 * k2 * fw * nc * rs + np.minimum(cfg.rprod * prod,
                                                      1.5 * cb2 * (gn[0][:C] ** 2 + gn[1][:C] ** 2) * ore)
    return res, src * vol[:C] - gather(conv) - gather(diff)
