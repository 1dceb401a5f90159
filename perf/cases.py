"""The workloads that this library's speed is measured on.

Every case is something a program that uses the library does over and over:
a simulation step, one multigrid V-cycle on its own arrays, a refinement
solve to a tolerance, a batch of solves, a batch of simulations, a burst of
served requests.  Sizes are those of the repository's own workloads, tests
and of the reference's default level, and odd or ragged ones beside them.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and handles, made from the seed
    run(state)           one pass through the public entry points
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    run()'s outputs in float64, in plain torch
"""
import math

import numpy as np
import torch

import ubootgl_amd as U
from ubootgl_amd import _lib as L
from ubootgl_amd.batch import Batch, SimBatch
from ubootgl_amd.serve import Server


def listed():
    return [
        # the smallest step: a thumbnail domain, all launches and latency
        step("step_64x32", 64, 32),
        # a small domain whose projection is solved well (10 V-cycles a step)
        step("step_512x256_10cycles", 512, 256, cycles=10),
        # the reference's default level: a channel between terrain, a thousand
        # tracers that the program reads back to draw them
        step("frame_1090x436", 1090, 436, scene="channel", tracers=1000, read_tracers=True),
        # an odd-sized step, neither side even
        step("step_1921x1081", 1921, 1081),
        # the headline simulation: 2/2 smoothing, a million tracers
        step("step_4096x2048", 4096, 2048, nu=2, tracers=1_000_000),
        # a step whose fields do not fit the last-level cache
        step("step_8192x4096", 8192, 4096),
        # one V-cycle on a program's own torch arrays (a preconditioner call),
        # at the odd size of the reference's multigrid test
        dict(name="vcycle_1025x1025", kind="vcycle", W=1025, H=1025, nu=3, zg=False),
        # refinement solves: an ordinary one to single accuracy, a large one to
        # the tolerance only the float64 residual reaches
        dict(name="solve_1024x512", kind="solve", W=1024, H=512, tol=1e-6),
        dict(name="solve_8192x4096", kind="solve", W=8192, H=4096, tol=1e-10),
        # two dozen unequal domains solved together
        dict(name="batch_24", kind="batch", n=24, lo=128, hi=1024, tol=1e-6),
        # sixteen unequal simulations stepped together
        dict(name="sims_16", kind="sims", n=16, lo=128, hi=1024),
        # a burst of requests, three warm-started solves each
        dict(name="serve_12", kind="serve", n=12, lo=64, hi=1024, tol=1e-6),
    ]


def step(name, W, H, nu=3, cycles=2, scene="walls", tracers=0, read_tracers=False, mu=0.001):
    return dict(name=name, kind="step", W=W, H=H, nu=nu, cycles=cycles, scene=scene,
                tracers=tracers, read_tracers=read_tracers, mu=mu)


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step"] * 5 + ["vcycle", "solve", "solve", "batch", "sims", "serve"])
    if kind == "step":
        W = logint(40, 8192)
        H = max(24, min(4096, int(W / rng.uniform(0.8, 4.0))))
        tracers = rng.choice([0, logint(100, 1_000_000)])
        c = step("", W, H, nu=rng.choice([2, 3]), cycles=rng.choice([1, 2, 2, 4]),
                 scene=rng.choice(["walls", "channel"]), tracers=tracers,
                 read_tracers=tracers < 5000 and rng.random() < 0.5,
                 mu=rng.choice([0.001, 0.0001]))
        del c["name"]
        return c
    if kind == "vcycle":
        W = logint(64, 1600)
        return dict(kind=kind, W=W, H=max(32, min(1600, int(W / rng.uniform(0.8, 3.0)))),
                    nu=rng.choice([2, 3]), zg=rng.random() < 0.5)
    if kind == "solve":
        W = logint(96, 4096)
        return dict(kind=kind, W=W, H=max(64, int(W / rng.uniform(1.0, 3.0))),
                    tol=rng.choice([1e-6, 1e-8, 1e-10]))
    lo = rng.choice([64, 128])
    return dict(kind=kind, n=rng.randint(4, 20), lo=lo, hi=rng.randint(300, 1024),
                **({} if kind == "sims" else {"tol": 1e-6}))


# ---- inputs ----------------------------------------------------------------

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def obstacles(W, H, g, scene):
    """Flag (1 = fluid) as a float32 tensor: disks, one at most in each cell of
    a lattice and clear of its edges (so that no pocket of fluid is closed
    off), about 5% of the area.  scene: 'open' leaves the outer ring fluid,
    'walls' closes it, 'channel' has rolling terrain along the two long sides
    and open ends."""
    P = int(min(256, max(16, min(W, H) // 4)))
    nx, ny = W // P + 1, H // P + 1
    r = np.where(g.random((ny, nx)) < 0.5, P * 0.06 * 6.0 ** g.random((ny, nx)), -1.0)
    cx = (np.arange(nx) + 0.5) * P + g.uniform(-0.12, 0.12, (ny, nx)) * P
    cy = (np.arange(ny)[:, None] + 0.5) * P + g.uniform(-0.12, 0.12, (ny, nx)) * P
    cx, cy, r2 = (torch.tensor(a, device=DEV) for a in (cx, cy, np.where(r > 0, r * r, -1.0)))
    x, y = torch.arange(W, device=DEV), torch.arange(H, device=DEV)
    i, j = (x // P)[None, :], (y // P)[:, None]
    d2 = (x[None, :] - cx[j, i]) ** 2 + (y[:, None] - cy[j, i]) ** 2
    fl = (d2 > r2[j, i]).to(torch.float32)
    if scene == "channel":
        X = torch.arange(W, device=DEV, dtype=torch.float64) / W
        for side in (0, 1):
            a = sum(math.pi ** -k * torch.sin(2 * math.pi * (k + 1) * X * W / H +
                                              float(g.uniform(0, 6.28))) for k in range(4))
            depth = (H * (0.11 + 0.07 * a)).clamp(min=1.0)[None, :]
            dist = y[:, None] if side == 0 else (H - 1 - y)[:, None]
            fl[dist < depth] = 0.0
    if scene == "open":
        fl[:2, :] = fl[-2:, :] = 1.0
        fl[:, :2] = fl[:, -2:] = 1.0
    if scene == "walls":
        fl[0, :] = fl[-1, :] = 0.0
        fl[:, 0] = fl[:, -1] = 0.0
    return fl


def modes(shape, x0, y0, W, H, g, n=8):
    """Sum of n sinusoidal modes with wavenumbers 1..6, random phases, float64
    (sin(a + b) as a product of one-dimensional factors)."""
    X = (torch.arange(shape[1], device=DEV, dtype=torch.float64) + x0) / W * 2 * math.pi
    Y = (torch.arange(shape[0], device=DEV, dtype=torch.float64) + y0) / H * 2 * math.pi
    k = torch.tensor(g.integers(1, 7, (2, n)), device=DEV, dtype=torch.float64)
    ph = torch.tensor(g.uniform(0, 2 * math.pi, n), device=DEV)
    a, b = k[0][:, None] * X[None, :] + ph[:, None], k[1][:, None] * Y[None, :]
    return torch.sin(b).T @ torch.cos(a) + torch.cos(b).T @ torch.sin(a)


def velocity(fl, g):
    H, W = fl.shape
    F = fl.double()
    vx = modes((H, W - 1), 0.5, 0.0, W, H, g) * F[:, :-1] * F[:, 1:]
    vy = modes((H - 1, W), 0.0, 0.5, W, H, g) * F[:-1, :] * F[1:, :]
    return vx, vy


def sim_inputs(case, seed):
    """Flag, the velocity as a new simulation holds it, and dt at CFL 0.5."""
    W, H = case["W"], case["H"]
    g = np.random.default_rng(seed)
    fl = obstacles(W, H, g, case["scene"])
    vx, vy = (v.float() for v in velocity(fl, g))
    vmax = max(float(vx.abs().max()), float(vy.abs().max()), 1e-3)
    vx[:, 0] = 1.0
    vy[0, :] = 0.0
    pwidth = np.float32((W - 1) / W)
    h = np.float32(pwidth / np.float32(W - 1))
    dt = np.float32(0.5 * float(h) / vmax)
    xy = None
    if case["tracers"]:
        n, f = case["tracers"], fl.cpu().numpy()
        x, y = g.uniform(2, W - 2, 4 * n), g.uniform(2, H - 2, 4 * n)
        ok = f[y.astype(int), x.astype(int)] > 0.5
        xy = np.stack([x[ok][:n], y[ok][:n]], 1) * (float(pwidth) / W)
    return dict(flag=fl, vx=vx, vy=vy, pwidth=pwidth, h=h, dt=dt, xy=xy)


def new_sim(case, inp):
    prm = U.Params(nu_pre=case["nu"], nu_post=case["nu"], vcycles_per_step=case["cycles"])
    sim = U.Simulation(inp["flag"].cpu().numpy(), inp["pwidth"], np.float32(case["mu"]), prm)
    vx, vy = inp["vx"].cpu().numpy(), inp["vy"].cpu().numpy()
    for k, v in (("vx", vx), ("vx_back", vx), ("vy", vy), ("vy_back", vy)):
        sim.set(k, v)
    if inp["xy"] is not None:
        sim.set_tracers(inp["xy"])
    return sim


def solve_inputs(W, H, g, steps=1):
    """Flag with a fluid outer ring, spacing, and `steps` right-hand sides: the
    divergence of a sinusoidal field whose second part grows step by step."""
    fl = obstacles(W, H, g, "open")
    h = float(np.float32(1.0 / W))
    va, vb = velocity(fl, g), velocity(fl, g)
    rhs = []
    for t in range(steps):
        vx, vy = (a + 0.25 * t * b for a, b in zip(va, vb))
        f = torch.zeros((H, W), device=DEV, dtype=torch.float64)
        f[1:-1, 1:-1] = -(vx[1:-1, 1:] - vx[1:-1, :-1] + vy[1:, 1:-1] - vy[:-1, 1:-1]) / h
        rhs.append((f * fl).float())
    return fl, rhs, h


def sizes(case, seed):
    """n unequal sizes, widths log-uniform in [lo, hi], aspect 1 to 4."""
    g = np.random.default_rng([seed, 1])
    out = []
    for _ in range(case["n"]):
        W = int(round(math.exp(g.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        out.append((W, max(32, int(W / g.uniform(1, 4)))))
    return out


def sims_cases(case):
    # sizes belong to the case, not to the seed: one plan, other inputs
    return [step("", W, H) for W, H in sizes(case, case["n"])]


class View:
    """A device field as the array interface that torch wraps without a copy.
    The tensor keeps this object, and with it the handle that owns the field."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(ptr, False),
                                             strides=None, version=2)


class Fields:
    """Torch views of a simulation's device fields, one for each buffer the
    fields move between."""

    def __init__(self, sim, names=("vx", "vy", "p")):
        self.sim, self.views = sim, {}
        self.names = [(n, L.FIELD_NAMES.index(n)) for n in names]

    def get(self):
        out = {}
        for name, fid in self.names:
            ptr = L.C.c_void_p()
            L.check(L.lib().ubg_sim_field_device_ptr(self.sim._h, fid, L.C.byref(ptr)))
            v = self.views.get((name, ptr.value))
            if v is None:
                v = torch.as_tensor(View(self.sim, ptr.value, self.sim.shape(name), "<f4"),
                                    device="cuda")
                self.views[name, ptr.value] = v
            out[name] = v
        return out


def prepare(case, seed):
    kind, g = case["kind"], np.random.default_rng(seed)
    st = dict(case=case)
    if kind == "step":
        inp = sim_inputs(case, seed)
        st.update(sim=new_sim(case, inp), dt=float(inp["dt"]), seed=seed & 0xffff)
        st["fields"] = Fields(st["sim"])
    elif kind == "sims":
        inps = [sim_inputs(c, seed * 1000 + i) for i, c in enumerate(sims_cases(case))]
        sims = [new_sim(c, i) for c, i in zip(sims_cases(case), inps)]
        st.update(batch=SimBatch(sims), fields=[Fields(s) for s in sims],
                  dts=np.array([i["dt"] for i in inps], np.float32))
    elif kind == "vcycle":
        fl, rhs, h = solve_inputs(case["W"], case["H"], g)
        prm = U.Params(nu_pre=case["nu"], nu_post=case["nu"])
        st.update(p=torch.zeros_like(rhs[0]), f=rhs[0], flag=fl.to(torch.uint8), h=h, prm=prm)
    elif kind == "solve":
        fl, rhs, h = solve_inputs(case["W"], case["H"], g)
        mg = U.MG(fl.cpu().numpy())
        mg.ir_set_rhs(rhs[0].cpu().numpy())
        st.update(mg=mg, h=h, views={})
    elif kind == "batch":
        b = Batch(sizes(case, case["n"]))
        for d, (W, H) in enumerate(b.sizes):
            fl, rhs, h = solve_inputs(W, H, g)
            b.set_domain(d, fl.cpu().numpy(), rhs[0].cpu().numpy(), h)
        st.update(batch=b)
    elif kind == "serve":
        srv = Server(hbm_budget=8 * 10**9, tol=case["tol"])
        reqs = []
        for W, H in sizes(case, case["n"]):
            fl, rhs, h = solve_inputs(W, H, g, steps=3)
            reqs.append((srv.add_geometry(fl.cpu().numpy(), h), [r.cpu().numpy() for r in rhs]))
        st.update(server=srv, reqs=reqs)
    return st


# ---- one pass --------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "step":
        sim = st["sim"]
        sim.step(st["dt"])
        if case["tracers"]:
            sim.advect_tracers(st["dt"], st["seed"])
        out = st["fields"].get()
        if case["read_tracers"]:
            out["tracers"], out["age"] = sim.get_tracers()
        return out
    if kind == "sims":
        st["batch"].step(st["dts"])
        return [f.get() for f in st["fields"]]
    if kind == "vcycle":  # one more V-cycle on the program's own arrays
        H, W = st["p"].shape
        L.check(L.lib().ubg_mg_solve_device_noalloc(
            st["p"].data_ptr(), st["f"].data_ptr(), st["flag"].data_ptr(), W, H, st["h"],
            int(case["zg"]), 1, L.C.byref(st["prm"]._p), torch.cuda.current_stream().cuda_stream))
        return st["p"]
    if kind == "solve":  # from a zero guess to the tolerance; the solution stays on the GPU
        mg = st["mg"]
        mg.ir_set_guess(None)
        mg.ir_solve(st["h"], tol=case["tol"])
        x = L.C.POINTER(L.C.c_double)()
        L.check(L.lib().ubg_mg_ir_device_ptrs(mg._h, L.C.byref(x), None))
        ptr = L.C.cast(x, L.C.c_void_p).value
        v = st["views"].get(ptr)
        if v is None:
            v = torch.as_tensor(View(mg, ptr, (case["H"], case["W"]), "<f8"), device="cuda")
            st["views"][ptr] = v
        return v
    if kind == "batch":
        b = st["batch"]
        for d in range(len(b)):
            b.set_guess(d)
        b.solve(tol=case["tol"])
        return [b.solution(d) for d in range(len(b))]
    if kind == "serve":
        srv = st["server"]
        ids = [srv.submit(gid, rhs, want_x=True) for gid, rhs in st["reqs"]]
        return [srv.wait(i)["x"] for i in ids]


# ---- what a pass cannot do without -----------------------------------------

def work(case):
    kind = case["kind"]

    def vcycle(nu):  # operations a cell of all levels: sweeps, residual, transfers
        return 4 / 3 * (2 * nu * 9 + 12 + 12)

    def step_work(c):
        n = c["W"] * c["H"]
        # vx, vy, p in and out, the saved velocity out, the flag in; a
        # tracer's position and age in and out
        b = n * (16 + 8 + 8 + 1) + 24 * c["tracers"]
        # diffuse 2 x 2 x 20, advect 2 faces x 3 samples x 5 cubics x 26,
        # divergence and correction 12; a tracer's two bilinear samples
        f = n * (80 + 820 + 12 + c["cycles"] * vcycle(c["nu"])) + 80 * c["tracers"]
        return b, f

    if kind == "step":
        b, f = step_work(case)
    elif kind == "sims":
        b, f = (sum(t) for t in zip(*map(step_work, sims_cases(case))))
    elif kind == "vcycle":
        n = case["W"] * case["H"]
        b, f = 13 * n, vcycle(case["nu"]) * n  # p in and out, f and flag in
    else:
        n = [(case["W"], case["H"])] if kind == "solve" else sizes(case, case["n"])
        n = sum(w * h for w, h in n) * (3 if kind == "serve" else 1)
        # right-hand side and flag in, float64 solution out; about six
        # V-cycles a decade
        b, f = 13 * n, 6 * math.log10(1 / case["tol"]) * vcycle(3) * n
    return {"bytes": float(b), "flops": float(f)}


# ---- the same in float64, in plain torch ------------------------------------

class Multigrid:
    """The V-cycle (red/black Gauss-Seidel, full weighting, flag-weighted
    prolongation) on float64 tensors."""

    def __init__(self, flag, h, nu=3, nu_coarse=5):
        self.nu, self.nu_coarse, self.lv = nu, nu_coarse, []
        F, h = flag.double(), float(h)
        while min(F.shape) > 3:
            H, W = F.shape
            s = F[1:-1, :-2] + F[1:-1, 2:] + F[2:, 1:-1] + F[:-2, 1:-1]
            inv = torch.where(s > 0, F[1:-1, 1:-1] / s.clamp(min=1), torch.zeros_like(s))
            y = torch.arange(1, H - 1, device=F.device)[:, None]
            x = torch.arange(1, W - 1, device=F.device)[None, :]
            self.lv.append(dict(F=F, inv=inv, odd=(x + y) % 2 == 1, h=h))
            Hc, Wc = H // 2, W // 2
            Fc = torch.ones((Hc, Wc), device=F.device, dtype=F.dtype)
            if min(Hc, Wc) > 2:
                Fc[1:-1, 1:-1] = (self.weigh(F, Wc, Hc) >= 4).double()
            h = h * (W - 1.0) / (Wc - 1.0) if Wc > 1 else h
            F = Fc

    @staticmethod
    def weigh(r, Wc, Hc):
        s = [[r[1 + j:2 * Hc - 3 + j + 1:2, 1 + i:2 * Wc - 3 + i + 1:2] for i in range(3)]
             for j in range(3)]
        s = [[t[:Hc - 2, :Wc - 2] for t in row] for row in s]
        return sum(t * ((2 if j == 1 else 1) * (2 if i == 1 else 1))
                   for j, row in enumerate(s) for i, t in enumerate(row))

    def sweep(self, lv, p, f):
        fhh = f[1:-1, 1:-1] * lv["h"] * lv["h"]
        for colour in (lv["odd"], ~lv["odd"]):
            q = p * lv["F"]
            val = q[1:-1, :-2] + q[1:-1, 2:] + q[:-2, 1:-1] + q[2:, 1:-1] + fhh
            c = p[1:-1, 1:-1]
            c.copy_(torch.where(colour, val * lv["inv"], c))

    def residual(self, lv, p, f):
        F, r = lv["F"], torch.zeros_like(p)
        pc, v = p[1:-1, 1:-1], 0
        for sl in ((slice(1, -1), slice(None, -2)), (slice(1, -1), slice(2, None)),
                   (slice(None, -2), slice(1, -1)), (slice(2, None), slice(1, -1))):
            v = v + F[sl] * (p[sl] - pc)
        r[1:-1, 1:-1] = (f[1:-1, 1:-1] + v / lv["h"] ** 2) * F[1:-1, 1:-1]
        return r

    @staticmethod
    def zero_gradient(p):
        p[1:-1, 0], p[1:-1, -1] = p[1:-1, 1].clone(), p[1:-1, -2].clone()
        p[0, 1:-1], p[-1, 1:-1] = p[1, 1:-1].clone(), p[-2, 1:-1].clone()

    def prolong(self, lv, lc, ec):
        F, Fc = lv["F"], lc["F"]
        H, W = F.shape
        e = torch.zeros_like(F)
        x2, y2 = torch.arange(2, W - 1, 2), torch.arange(2, H - 1, 2)
        x1, y1 = torch.arange(1, W - 2, 2), torch.arange(1, H - 2, 2)
        for ys in (y2, y1):
            for xs in (x2, x1):
                if not len(xs) or not len(ys):
                    continue
                jj = [ys // 2] + ([ys // 2 + 1] if ys is y1 else [])
                ii = [xs // 2] + ([xs // 2 + 1] if xs is x1 else [])
                sl = (slice(int(ys[0]), int(ys[-1]) + 1, 2), slice(int(xs[0]), int(xs[-1]) + 1, 2))
                cut = [(slice(int(j[0]), int(j[-1]) + 1), slice(int(i[0]), int(i[-1]) + 1))
                       for j in jj for i in ii]
                num = sum(ec[c] for c in cut)
                e[sl] = F[sl] * num / ((sum(Fc[c] for c in cut) + 0.0001) if len(cut) > 1 else 1)
        return e

    def cycle(self, p, f, zg=False, level=0):
        lv = self.lv[level]
        if level == len(self.lv) - 2:
            for _ in range(self.nu_coarse):
                self.sweep(lv, p, f)
            return
        zg = zg and level == 0
        for _ in range(self.nu):
            self.sweep(lv, p, f)
            if zg:
                self.zero_gradient(p)
        lc = self.lv[level + 1]
        Hc, Wc = lc["F"].shape
        fc = torch.zeros_like(lc["F"])
        fc[1:-1, 1:-1] = self.weigh(self.residual(lv, p, f), Wc, Hc) / 16
        ec = torch.zeros_like(fc)
        self.cycle(ec, fc, False, level + 1)
        e = self.prolong(lv, lc, ec)
        p[1:-1, 1:-1] += e[1:-1, 1:-1]
        if zg:
            self.zero_gradient(p)
        for _ in range(self.nu):
            self.sweep(lv, p, f)
            if zg:
                self.zero_gradient(p)

    def solve(self, f, tol, limit=120):
        """Float64 solution with the outer ring at zero, to a relative residual."""
        x, f = torch.zeros_like(f, dtype=torch.float64), f.double()
        f0 = float(torch.linalg.vector_norm(self.residual(self.lv[0], x, f)))
        for k in range(limit):
            self.cycle(x, f)
            if k % 4 == 3 and float(torch.linalg.vector_norm(
                    self.residual(self.lv[0], x, f))) <= tol * f0:
                break
        return x


class Step:
    """Simulation::step on float64 tensors with the default boundary kinds:
    inflow west, zero-pressure outflow east, no slip north and south."""

    def __init__(self, case, inp):
        self.case = case
        self.F = inp["flag"].double()
        self.vx = [inp["vx"].double().clone() for _ in range(2)]  # front, back
        self.vy = [inp["vy"].double().clone() for _ in range(2)]
        self.p = torch.zeros_like(self.F)
        self.h, self.dt, self.pw = float(inp["h"]), float(inp["dt"]), float(inp["pwidth"])
        self.mg = Multigrid(self.F, self.h, case["nu"])

    def vbcs(self):
        (x, xb), (y, yb) = self.vx, self.vy
        out = (lambda a: a.clamp(min=0))
        # west inflow keeps its value; east takes max(a, 0); the rest mirror or stop
        x[:, -1] = out(x[:, -2])
        x[0], x[-1] = -x[1], -x[-2]
        y[:, -1] = out(y[:, -2])
        y[0], y[-1] = 0.0, 0.0
        for f, b in ((x, xb), (y, yb)):
            b[0], b[-1], b[:, 0], b[:, -1] = f[0], f[-1], f[:, 0], f[:, -1]

    def diffuse(self):
        F, W = self.F, self.F.shape[1]
        a = self.dt * float(np.float32(self.case["mu"])) * (W - 1.0) / self.pw

        def jacobi(v, own, fe, fw, fn, fs):
            # v is indexed [across, along]: along-neighbours are masked, the
            # two beside mirrored where their face is blocked
            c = v[1:-1, 1:-1]
            s = v[1:-1, 2:] * fe + v[1:-1, :-2] * fw
            s = s + v[2:, 1:-1] * fn - (1 - fn) * c + v[:-2, 1:-1] * fs - (1 - fs) * c
            return own * (c + a * s) / (1 + 4 * a)

        fx = F[:, :-1] * F[:, 1:]                # face (x, x+1)
        beside = F[:, :-1] * F[:, 1:]            # F(x-1) F(x), at column x - 1
        for _ in range(2):
            v = self.vx[0]
            self.vx[1][1:-1, 1:-1] = jacobi(v, fx[1:-1, 1:-1], fx[1:-1, 2:], fx[1:-1, :-2],
                                            beside[2:, :-2], beside[:-2, :-2])
            self.vx.reverse()
            self.vbcs()
        fy = (F[:-1] * F[1:]).T                  # face (y, y+1), transposed
        for _ in range(2):
            v = self.vy[0]
            # beside: F(x+-1, y) F(x+-1, y+1), the neighbouring columns' faces
            new = jacobi(v.T, fy[1:-1, 1:-1], fy[1:-1, 2:], fy[1:-1, :-2], fy[2:, 1:-1],
                         fy[:-2, 1:-1])
            self.vy[1][1:-1, 1:-1] = new.T
            self.vy.reverse()
            self.vbcs()

    @staticmethod
    def cubic(t, A, B, C, D):
        a = -A / 2 + 3 * B / 2 - 3 * C / 2 + D / 2
        b = A - 5 * B / 2 + 2 * C - D / 2
        return ((a * t + b) * t + (C - A) / 2) * t + B

    @classmethod
    def sample(cls, g, cx, cy):
        H, W = g.shape
        cx, cy = cx.clamp(3.0, W - 3.0), cy.clamp(3.0, H - 3.0)
        ix, iy = cx.long(), cy.long()
        base = (iy - 1) * W + ix - 1
        sx, sy, g = cx - ix, cy - iy, g.reshape(-1)
        col = [cls.cubic(sy, *(g[base + (k * W + m)] for k in range(4))) for m in range(4)]
        return cls.cubic(sx, *col)

    def advect(self):
        F, (H, W) = self.F, self.F.shape
        xf, yf = self.vx[0], self.vy[0]
        k = self.dt / self.h
        new = [self.vx[1].clone(), self.vy[1].clone()]
        for vertical in (False, True):
            w = W if vertical else W - 1
            nck = max(0, (w - 9 + 7) // 8)       # chunks of 8 from x = 1, clear of the edge
            if not nck:
                continue
            y = torch.arange(1, H - 1, device=F.device)[:, None]
            x = torch.arange(1, 8 * nck + 1, device=F.device)[None, :]
            other = F[y - 1, x] if vertical else F[y, x - 1]
            live = (F[y, x] * other).reshape(H - 2, nck, 8).amax(-1) > 0
            live = live.repeat_interleave(8, 1)
            X, Y = xf.reshape(-1), yf.reshape(-1)
            xi, yi = y * (W - 1) + x, y * W + x  # flat: a row's end runs into the next
            if vertical:
                u = (X[xi] + X[xi - W + 1] + X[xi + 1] + X[xi - W + 2]) / 4
                v, px, py = Y[yi], x.double(), y + 0.5
            else:
                v = (Y[yi] + Y[yi - W] + Y[yi + 1] + Y[yi - W + 1]) / 4
                u, px, py = X[xi], x + 0.5, y.double()
            mx, my = px - u * (k / 2), py - v * (k / 2)
            u, v = self.sample(xf, mx - 0.5, my), self.sample(yf, mx, my - 0.5)
            ex, ey = px - u * k, py - v * k
            if vertical:
                val = self.sample(yf, ex, ey - 0.5) * F[y, x] * F[y + 1, x]
            else:
                val = self.sample(xf, ex - 0.5, ey) * F[y, x] * F[y, x + 1]
            to = new[vertical][1:H - 1, 1:8 * nck + 1]
            to.copy_(torch.where(live, val, to))
        self.vx, self.vy = [new[0], xf], [new[1], yf]

    def project(self):
        F, p, ih = self.F, self.p, 1 / self.h
        x, y = self.vx[0], self.vy[0]
        f = torch.zeros_like(p)
        f[1:-1, 1:-1] = -ih * (x[1:-1, 1:] - x[1:-1, :-1] + y[1:, 1:-1] - y[:-1, 1:-1])
        for _ in range(self.case["cycles"]):
            self.mg.cycle(p, f, zg=True)
        p[:, 0], p[:, -1] = p[:, 1].clone(), -p[:, -2]
        p[0], p[-1] = p[1].clone(), p[-2].clone()
        x[1:-1, 1:-1] -= (F[:, :-1] * F[:, 1:] * ih * (p[:, 1:] - p[:, :-1]))[1:-1, 1:-1]
        y[1:-1, 1:-1] -= (F[:-1] * F[1:] * ih * (p[1:] - p[:-1]))[1:-1, 1:-1]

    def step(self):
        self.diffuse()
        self.advect()
        self.vbcs()
        self.project()
        self.vbcs()
        return dict(vx=self.vx[0], vy=self.vy[0], p=self.p)


def exact(case, seed):
    kind, g = case["kind"], np.random.default_rng(seed)
    if kind == "step":
        out = Step(case, sim_inputs(case, seed)).step()
        if case["read_tracers"]:  # respawns and cell tests are not a smooth function
            out["tracers"], out["age"] = None, None
        return out
    if kind == "sims":
        return [Step(c, sim_inputs(c, seed * 1000 + i)).step()
                for i, c in enumerate(sims_cases(case))]
    if kind == "vcycle":
        fl, rhs, h = solve_inputs(case["W"], case["H"], g)
        p = torch.zeros_like(rhs[0], dtype=torch.float64)
        Multigrid(fl, h, case["nu"]).cycle(p, rhs[0].double(), zg=case["zg"])
        return p
    if kind == "solve":
        fl, rhs, h = solve_inputs(case["W"], case["H"], g)
        return Multigrid(fl, h).solve(rhs[0], case["tol"] * 1e-3)
    steps = 3 if kind == "serve" else 1
    out = []
    for W, H in sizes(case, case["n"]):
        fl, rhs, h = solve_inputs(W, H, g, steps=steps)
        out.append(Multigrid(fl, h).solve(rhs[-1], case["tol"] * 1e-3))
    return out
