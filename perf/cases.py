"""Workloads of the time step, the ensemble and the adjoint, for timing.

listed() names the workloads, draw() gives more of the same ranges; prepare()
builds one from a seed, run() is one pass of it through the public entry
points, work() the bytes and operations a pass cannot do without and exact()
its outputs as a plain 64-bit torch program computes them.

Three kinds of pass:

steps     a stretch of a simulation: r3d_hip_step over `steps` RK3 steps, then
          the state dumped into the program's own pinned host buffers (a run
          that writes its fields every `steps` steps).  The state lives on in
          the context, so each pass goes on where the last one ended.
ensemble  the same for many independent members (r3d_ens_step).
adjoint   one evaluation of the final kinetic energy and its gradient with
          respect to the initial temperature, Re and theta, through the torch
          binding (the inner call of an optimisation).
"""
import ctypes
import importlib

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

from __graft_entry__ import load_package

pkg = load_package()
PRIMARIES = ["ru", "rv", "rw", "ro", "tt", "bx", "by", "bz"]

# Physics of the repository's benchmark and tests, as host set-up flags.
ROT = ["--lrot", "1", "--ry", "0.1", "--ang", "0"]
PHYSICS = {
    "hydro": [],  # the default: a cold plume at the top wall
    "convection": ["--tp", "0"],  # no plume (on coarse grids the plume drives T below zero)
    "rotating": ROT,
    "mhd": ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp",
            "10"] + ROT,
    "heat": ["--itcon", "2", "--tp", "1.5", "--zp", "20.0", "--hh", "4.0"],
    "density": ["--ngrid", "0", "--id", "1", "--dh", "0.4", "--dv", "0.3"],
    "relax": ["--ngrid", "0", "--itcon", "0", "--izcon", "1", "--rlax", "0.5", "--toff", "0.5",
              "--tstart", "-1"],
}
# Relative cost of a cell-step of each kind, for the size limit of draw().
COST = {"hydro": 1.0, "convection": 1.0, "rotating": 1.0, "mhd": 2.1, "heat": 1.1, "density": 1.3, "relax": 1.9}
MOST = 504 * 504 * 256 * 50  # hydro cell-steps of the largest listed case


def case(name, kind, physics, npx, npy, npz, npey, npez, steps, variant=0, members=0):
    return {"name": name, "kind": kind, "physics": physics, "npx": npx, "npy": npy, "npz": npz,
            "npey": npey, "npez": npez, "steps": steps, "variant": variant, "members": members}


def listed():
    return [
        # the smallest grid in use (the smoke run's): launch latency
        case("hydro_16x16x32", "steps", "convection", 16, 16, 32, 2, 2, 100),
        # the reference's small configuration, a laptop-size run of 100 steps
        case("hydro_64x64x128", "steps", "hydro", 64, 64, 128, 1, 2, 100),
        # a ragged grid: partial tiles in x and y, a short last z chunk
        case("hydro_150x93x210", "steps", "rotating", 150, 93, 210, 3, 2, 50),
        # the production cross-section, on the 256 planes of the CPU baseline's sample
        case("hydro_504x504x256", "steps", "hydro", 504, 504, 256, 4, 2, 50),
        # the FMA-contracted variant on a medium grid
        case("fma_252x252x256", "steps", "hydro", 252, 252, 256, 2, 4, 50, variant=1),
        # MHD: a small ragged grid and the rotating-MHD benchmark grid
        case("mhd_100x70x90", "steps", "mhd", 100, 70, 90, 2, 3, 50),
        case("mhd_252x252x512", "steps", "mhd", 252, 252, 512, 2, 4, 30),
        # physics beyond the plain step that needs horizontal means every stage
        case("density_252x252x512", "steps", "density", 252, 252, 512, 4, 2, 30),
        case("relax_252x252x512", "steps", "relax", 252, 252, 512, 4, 2, 20),
        # the seeded ensemble workload: 64 members of uneven sizes
        case("ensemble_64", "ensemble", "hydro", 0, 0, 0, 1, 2, 30, members=64),
        # gradients on the adjoint benchmark grid, hydrodynamic and MHD
        case("adjoint_hydro_128x128x256", "adjoint", "hydro", 128, 128, 256, 2, 4, 20),
        case("adjoint_mhd_128x128x256", "adjoint", "mhd", 128, 128, 256, 2, 4, 20),
    ]


def draw(rng):
    def log_uniform(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    def ranks(n, most, least):
        return rng.choice([q for q in range(1, most + 1) if n % q == 0 and n // q >= least])

    kind = rng.choice(["steps", "steps", "steps", "adjoint", "adjoint", "ensemble"])
    if kind == "ensemble":
        return case("", kind, "hydro", 0, 0, 0, 1, 2, rng.randint(10, 30),
                    members=rng.randint(4, 48))
    while True:
        physics = rng.choice(["hydro", "mhd"] if kind == "adjoint" else sorted(PHYSICS))
        big = kind == "steps"
        small = physics == "convection"
        npx = log_uniform(16 if small else 24, 504 if big else 128)
        npy = log_uniform(12 if small else 20, 504 if big else 128)
        npz = log_uniform(32 if small else 48, 512 if big else 256)
        steps = rng.randint(10, 50) if big else rng.randint(4, 20)
        if COST[physics] * npx * npy * npz * steps > (MOST / 2 if big else MOST):
            continue
        npey = ranks(npy, 4, 3)
        npez = ranks(npz, 4, 3)
        if physics == "relax" and npez < 2:  # the relaxation needs two z ranks
            continue
        variant = int(physics in ("hydro", "convection", "rotating", "mhd") and big and rng.random() < 0.2)
        return case("", kind, physics, npx, npy, npz, npey, npez, steps, variant=variant)


def flags(c, seed):
    return ["--npx", str(c["npx"]), "--npy", str(c["npy"]), "--npz", str(c["npz"]), "--npey",
            str(c["npey"]), "--npez", str(c["npez"]), "--seed",
            str(-(1 + seed % 1000000))] + PHYSICS[c["physics"]]


def member_flags(c, seed):
    out = pkg.ensemble_members(c["members"], seed=3)
    for m, f in enumerate(out):
        f[f.index("--seed") + 1] = str(-(1 + (seed * 64 + m) % 1000000))
    return out


def perturbed(tt, seed):
    """The adjoint's initial temperature: the run's own, with a random part."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tt * (1.0 + 1e-3 * torch.randn(tt.shape, dtype=tt.dtype, device="cuda", generator=g))


def pinned(shapes):
    """Dense host arrays in one pinned buffer, and their addresses."""
    flat = torch.empty(sum(int(np.prod(s)) for s in shapes), dtype=torch.float64, pin_memory=True)
    out, at = [], 0
    for s in shapes:
        n = int(np.prod(s))
        out.append(flat[at:at + n].view(*s))
        at += n
    return flat, out


def pointers(arrays):
    p = ctypes.POINTER(ctypes.c_double)
    a = (p * 16)()
    for q, x in enumerate(arrays):
        a[q] = ctypes.cast(x.data_ptr(), p)
    return a


def prepare(c, seed):
    if c["kind"] == "adjoint":
        at = importlib.import_module("rast3dmhd_amd.adjoint_torch")
        prob = at.KineticEnergyRun(flags(c, seed), c["steps"])
        prob.adjoint(prob.cfg.re, prob.cfg.theta)  # the context it keeps on the GPU
        one = dict(dtype=torch.float64, device="cuda")
        return {"kind": "adjoint", "prob": prob,
                "tt": perturbed(prob.initial_tt().cuda(), seed).requires_grad_(True),
                "re": torch.tensor(prob.cfg.re, requires_grad=True, **one),
                "theta": torch.tensor(prob.cfg.theta, requires_grad=True, **one)}
    if c["kind"] == "ensemble":
        runs = [pkg.Run(f) for f in member_flags(c, seed)]
        sim = pkg.Ensemble(runs)
        sim.autotune(3)
        shapes = [r.shape for r in runs for _ in range(5)]
        for r in runs:
            r.close()
        flat, arrays = pinned(shapes)
        return {"kind": "ensemble", "sim": sim, "steps": c["steps"], "flat": flat,
                "to": [pointers(arrays[5 * m:5 * m + 5]) for m in range(len(runs))]}
    run_ = pkg.Run(flags(c, seed))
    sim = run_.make_sim(c["variant"])
    flat, arrays = pinned([run_.shape] * sim.nf)
    run_.close()
    return {"kind": "steps", "sim": sim, "steps": c["steps"], "fields": arrays,
            "to": pointers(arrays)}


def check(rc):
    if rc != 0:
        raise RuntimeError(pkg.load().r3d_hip_last_error().decode())


def run(s):
    if s["kind"] == "adjoint":
        for q in ("tt", "re", "theta"):
            s[q].grad = None
        J = s["prob"](s["tt"], s["re"], s["theta"])
        J.backward()
        return {"J": J.detach(), "tt": s["tt"].grad, "re": s["re"].grad, "theta": s["theta"].grad}
    s["sim"].step(s["steps"])
    if s["kind"] == "ensemble":
        for m, to in enumerate(s["to"]):
            check(pkg.load().r3d_ens_download_global(s["sim"].h, m, to))
        return s["flat"]
    check(pkg.load().r3d_hip_download_global(s["sim"].h, s["to"]))
    sc = s["sim"].scalars()
    return {"fields": s["fields"], "dt": sc["dt"], "timt": sc["timt"], "umach": sc["umach"]}


def cells_of(c):
    if c["kind"] != "ensemble":
        return c["npx"] * c["npy"] * c["npz"]
    total = 0
    for f in pkg.ensemble_members(c["members"], seed=3):
        total += int(f[1]) * int(f[3]) * int(f[5])
    return total


def work(c):
    """A step is three stages, each a function of the whole state: stage 1
    reads X and writes X' and the RK accumulator, stage 2 reads both and
    writes both, stage 3 reads both and writes X' (10 passes over the fields).
    Horizontal means are functions of a whole plane, so they read their field
    (density: ro; relaxation: tt, then all five) before the stage.  The
    adjoint adds, per stage, the state and the two adjoint fields read and
    one written.  Operations: those of the flux formulas."""
    mag = c["physics"] == "mhd"
    nf = 8 if mag else 5
    n = cells_of(c) * c["steps"]
    flops = 3 * (600 if mag else 370) * n
    b = 10 * nf * 8 * n
    if c["physics"] == "density":
        b += 3 * 8 * n
    if c["physics"] == "relax":
        b += 3 * 6 * 8 * n
    if c["kind"] == "adjoint":
        return {"bytes": b + 3 * 4 * nf * 8 * n, "flops": 4 * flops}
    return {"bytes": b + cells_of(c) * nf * 8, "flops": flops}


# ---- the same results in plain torch ---------------------------------------------------------
class Plain:
    """The RK3 step of one run on torch tensors (npz + 2, npy, npx), float64:
    x and y periodic, the two outer z planes fixed except for the density,
    which the step replaces by its reciprocal every stage."""

    def __init__(self, run_, device="cuda"):
        self.c = c = run_.cfg()
        m = {k: torch.from_numpy(np.array(v)).to(device) for k, v in run_.metrics().items()}
        x = y = z = slice(1, -1)
        self.x = {k: m[k][x].view(1, 1, -1) for k in ("dxxdx", "d2xxdx2", "ddx", "exx")}
        self.y = {k: m[k][y].view(1, -1, 1) for k in ("dyydy", "d2yydy2", "ddy", "wyy")}
        self.z = {k: m[k][z].view(-1, 1, 1)
                  for k in ("dzzdz", "d2zzdz2", "ddz", "rkapa", "dkapa", "zee")}
        self.nf = 8 if c.lmag else 5
        self.re = torch.tensor(c.re, dtype=torch.float64, device=device)
        self.theta = torch.tensor(c.theta, dtype=torch.float64, device=device)
        full = run_.state(copy=False)
        self.full = [torch.from_numpy(np.array(full[f])).to(device) for f in PRIMARIES[:self.nf]]
        self.X = [f[:, 1:-1, 1:-1].clone() for f in self.full]
        self.hx, self.hy, self.hz = (c.hx * self.x["dxxdx"], c.hy * self.y["dyydy"],
                                     c.hz * self.z["dzzdz"])
        self.lx = (c.hx * self.x["d2xxdx2"], c.h2x * self.x["dxxdx"] ** 2)
        self.ly = (c.hy * self.y["d2yydy2"], c.h2y * self.y["dyydy"] ** 2)
        self.lz = (c.hz * self.z["d2zzdz2"], c.h2z * self.z["dzzdz"] ** 2)
        ln2 = float(np.float32(-4.0) * np.log(np.float32(2.0)))

        def gauss(at, centre):
            return torch.exp(ln2 / c.hh / c.hh * (at - centre) ** 2)

        if c.tp != 0.0 or c.itcon == 2:
            self.plume = (gauss(self.x["exx"], c.xp) / c.hh * gauss(self.y["wyy"], c.yp) /
                          c.hh)[0]
            self.sink = (c.tp * c.ocv * self.plume * gauss(self.z["zee"], c.zp) / c.hh
                         if c.itcon == 2 else None)

    # centred differences of a field with both outer planes
    def dx(self, f):
        return (torch.roll(f, -1, 2) - torch.roll(f, 1, 2)) * self.hx

    def dy(self, f):
        return (torch.roll(f, -1, 1) - torch.roll(f, 1, 1)) * self.hy

    def dz(self, f):
        return (f[2:] - f[:-2]) * self.hz

    def laps(self, f):
        i = f[1:-1]
        e, w = torch.roll(i, -1, 2), torch.roll(i, 1, 2)
        n, s = torch.roll(i, -1, 1), torch.roll(i, 1, 1)
        u, d = f[2:], f[:-2]
        return ((e - w) * self.lx[0] + (e - 2.0 * i + w) * self.lx[1],
                (n - s) * self.ly[0] + (n - 2.0 * i + s) * self.ly[1],
                (u - d) * self.lz[0] + (u - 2.0 * i + d) * self.lz[1])

    def fluxes(self, X, re):
        c = self.c
        ru, rv, rw, ro, tt = X[:5]
        ri = 1.0 / ro
        u, v, w, p = ru * ri, rv * ri, rw * ri, ro * tt
        I = slice(1, -1)  # the planes of the domain
        ore, tk = 1.0 / re, c.ocv / (re * (c.repr / c.re))
        t1, t2, t3 = c.ocv * ore, c.c13 * ore, c.c43 * c.ocv * ore
        dx, dy, dz, R = self.dx, self.dy, self.dz, ri[I]

        rwz = torch.cat([(4.0 * rw[2:3] - rw[3:4]) * self.hz[:1], dz(rw)[1:-1],
                         (rw[-4:-3] - 4.0 * rw[-3:-2]) * self.hz[-1:]])
        fr = -dx(ru[I]) - dy(rv[I]) - rwz
        if c.id == 1:
            pert = torch.cat([ro[2:3], ro[I], ro[-3:-2]])
            pert = pert - pert.mean((1, 2), keepdim=True)
            lap = self.laps(pert)
            wz = ore / ro[I].mean((1, 2), keepdim=True)
            fr = fr + c.dh * wz * (lap[0] + lap[1]) + c.dv * wz * lap[2]
        ux, uy, uz = dx(u[I]), dy(u[I]), dz(u)
        vx, vy, vz = dx(v[I]), dy(v[I]), dz(v)
        wx, wy, wz = dx(w[I]), dy(w[I]), dz(w)
        lu, lv, lw = self.laps(u), self.laps(v), self.laps(w)

        def adv(m):
            return dx((m * u)[I]) + dy((m * v)[I]) + dz(m * w)

        fu = -dx(p[I]) - adv(ru) + ore * (c.c43 * lu[0] + lu[1] + lu[2]) + t2 * (dy(vx) + dx(wz))
        fv = -dy(p[I]) - adv(rv) + ore * (lv[0] + c.c43 * lv[1] + lv[2]) + t2 * (dy(ux) + dy(wz))
        fw = (c.grav * ro[I] - dz(p) - adv(rw) + ore * (lw[0] + lw[1] + c.c43 * lw[2]) +
              t2 * (dx(uz) + dy(vz)))
        if c.lrot:
            fu = fu + c.omz * rv[I]
            fv = fv - c.omz * ru[I] + c.omx * rw[I]
            fw = fw - c.omx * rv[I]
        T, lt = tt[I], self.laps(tt)
        ft = -u[I] * dx(T) - v[I] * dy(T) - w[I] * dz(tt)
        ft = ft + ((lt[0] + lt[1] + lt[2]) * self.z["rkapa"] + dz(tt) * self.z["dkapa"]) * R * tk
        ft = ft + (c.c43 * ux * ux + vx * vx + wx * wx + uy * uy + 2.0 * uy * vx + uz * uz +
                   vz * vz + wy * wy + 2.0 * vz * wy + 2.0 * uz * wx) * R * t1
        ft = ft + (vy * vy + wz * wz - ux * wz - ux * vy - vy * wz) * R * t3
        ft = ft - c.ocv * (ux + vy + wz) * T
        if c.itcon == 2:
            ft = ft - self.sink * R
        if not c.lmag:
            return [fu, fv, fw, fr, ft]
        bx, by, bz = X[5:]
        bxy, byx, bzx, bxz = dy(bx[I]), dx(by[I]), dx(bz[I]), dz(bx)
        byz, bzy = dz(by), dy(bz[I])
        BX, BY, BZ, U, V, W = bx[I], by[I], bz[I], u[I], v[I], w[I]
        ob = c.obeta
        fu = fu + ob * (BY * (bxy - byx) - BZ * bzx + BZ * bxz)
        fv = fv + ob * (BX * (byx - bxy) + BZ * (byz - bzy))
        fw = fw + ob * (BX * bzx - BX * bxz - BY * (byz - bzy))
        ft = ft + ((bxy - byx) ** 2 + bzx * bzx + bxz * bxz - 2.0 * bxz * bzx +
                   (byz - bzy) ** 2) * R * (ob * c.orm * c.ocv)

        # one-sided z stencils on the walls (the bottom one with npez > 1)
        def walls(mid, top, bottom):
            return torch.cat([top, mid[1:-1], bottom if c.npez > 1 else mid[-1:]])

        wzm = walls(wz, (4.0 * w[2:3] - w[3:4]) * self.hz[:1],
                    (w[-4:-3] - 4.0 * w[-3:-2]) * self.hz[-1:])

        def lapz(f, mid):
            a, b, d, e = f[1:2], f[2:3], f[3:4], f[4:5]
            A, B, D, E = f[-2:-1], f[-3:-2], f[-4:-3], f[-5:-4]
            return walls(mid,
                         (-3.0 * a + 4.0 * b - d) * self.lz[0][:1] +
                         (2.0 * a - 5.0 * b + 4.0 * d - e) * self.lz[1][:1],
                         (3.0 * A - 4.0 * B + D) * self.lz[0][-1:] +
                         (2.0 * A - 5.0 * B + 4.0 * D - E) * self.lz[1][-1:])

        lbx, lby, lbz = self.laps(bx), self.laps(by), self.laps(bz)
        f1 = (BY * uy - BX * vy + BZ * uz - BX * wzm - U * dx(BX) - V * bxy - W * bxz +
              c.orm * (lbx[0] + lbx[1] + lapz(bx, lbx[2])))
        f2 = (BX * vx - BY * ux + BZ * vz - BY * wzm - U * byx - V * dy(BY) - W * byz +
              c.orm * (lby[0] + lby[1] + lapz(by, lby[2])))
        f3 = (BX * wx - BZ * ux + BY * wy - BZ * vy - U * bzx - V * bzy - W * dz(bz) +
              c.orm * (lbz[0] + lbz[1] + lbz[2]))
        return [fu, fv, fw, fr, ft, f1, f2, f3]

    def walls(self, X, theta):
        """The boundary conditions on planes 1 and npz."""
        c = self.c

        def side(f, k):
            return [f[k], f[k + (1 if k > 0 else -1)], f[k + (2 if k > 0 else -2)]]

        out = []
        ends = {}
        for k, top in ((1, True), (-2, False)):
            ro = side(X[3], k)
            m = [ro[0] * (c.c43 * f[1] / ro[1] - c.c13 * f[2] / ro[2])
                 for f in (side(X[0], k), side(X[1], k))]
            t = side(X[4], k)
            ext = c.c43 * t[1] - c.c13 * t[2]
            if top:
                dz = c.dzf / self.z["dzzdz"][0]
                if c.tp != 0.0 and c.itcon == 0:
                    tt = 1.0 - (1.0 - c.tp) * self.plume
                elif c.tp != 0.0 and c.itcon == 1:
                    tt = ext - c.c23 * dz * (theta - (theta - c.tp) * self.plume)
                elif c.itcon in (0, 2):
                    tt = torch.ones_like(t[0])
                else:
                    tt = ext - c.c23 * dz * theta
            else:
                dz = c.dzf / self.z["dzzdz"][-1]
                tt = (torch.full_like(t[0], c.tb) if c.izcon == 0
                      else ext + c.c23 * dz * theta / self.z["rkapa"][-1])
            ends[top] = m + [torch.zeros_like(t[0]), None, tt, None, None,
                             torch.zeros_like(t[0]) if c.ibcon == 0 else None]
        for q, f in enumerate(X):
            a, b = ends[True][q], ends[False][q]
            out.append(f if a is None else torch.cat([f[:1], a[None], f[2:-2], b[None], f[-1:]]))
        return out

    def limits(self, X, re):
        c = self.c
        ru, rv, rw, ro, tt = (f[1:-1] for f in X[:5])
        dd = torch.minimum(torch.minimum(self.x["ddx"], self.y["ddy"]), self.z["ddz"])
        uu = (ru * ru + rv * rv + rw * rw) / (ro * ro)
        a = c.gamma * tt
        if c.lmag:
            a = a + sum(f[1:-1] * f[1:-1] for f in X[5:]) * c.obeta / ro
        fast = uu + a + 2.0 * torch.sqrt(uu * a)
        pr = c.repr / c.re
        lim = [dd / torch.sqrt(fast), 0.5 * dd * dd * (re * pr) * c.cv * ro / self.z["rkapa"],
               0.375 * dd * dd * re * ro]
        if c.lmag:
            lim.append((0.5 * dd * dd * c.rm).expand_as(ro))
        # a cell where T fell below zero sets no limit (its fast speed is no number)
        return [torch.nan_to_num(q, nan=1e300) for q in lim], uu / tt / c.gamma

    def dt(self, X, re):
        with torch.no_grad():
            lim, _ = self.limits(X, re)
            least = [float(q.min()) for q in lim]
            which = least.index(min(least))
            at = int(lim[which].argmin())
        n = [int(q) for q in np.unravel_index(at, lim[which].shape)]
        # the limit at the cell that attains it
        c = self.c
        dd = torch.minimum(torch.minimum(self.x["ddx"].view(-1)[n[2]], self.y["ddy"].view(-1)[n[1]]),
                           self.z["ddz"].view(-1)[n[0]])
        ru, rv, rw, ro, tt = (f[n[0] + 1, n[1], n[2]] for f in X[:5])
        if which == 0:
            uu = (ru * ru + rv * rv + rw * rw) / (ro * ro)
            a = c.gamma * tt
            if c.lmag:
                a = a + sum(f[n[0] + 1, n[1], n[2]] ** 2 for f in X[5:]) * c.obeta / ro
            fast = uu + a + 2.0 * torch.sqrt(uu * a) if float(uu) > 0.0 else uu + a
            return c.sff * dd / torch.sqrt(fast)
        if which == 1:
            rk = self.z["rkapa"].view(-1)[n[0]]
            return c.sff * (0.5 * dd * dd * (re * (c.repr / c.re)) * c.cv * ro / rk)
        if which == 2:
            return c.sff * (0.375 * dd * dd * re * ro)
        return c.sff * (0.5 * dd * dd * c.rm)

    def stage(self, X, Z, dt, re, theta, s):
        """(X', Z') of one stage; Z = X in the first."""
        c = self.c
        gam, zeta = (c.gam1, c.gam2, c.gam3)[s], (c.zeta1, c.zeta2, 0.0)[s]
        F = self.fluxes(X, re)
        new = []
        for q in range(self.nf):
            x = Z[q][1:-1] + gam * dt * F[q]
            ends = [X[q][:1], X[q][-1:]]
            if q == 3:  # density diffusion mirrors the outer planes of ro before the fluxes
                ends = [X[q][2:3], X[q][-3:-2]] if c.id else ends
                ends = [1.0 / e for e in ends]
            new.append(torch.cat([ends[0], x, ends[1]]))
        new = self.walls(new, theta)
        mix = [f.clone() if s == 2 else torch.cat([f[:1], f[1:-1] + zeta * dt * g, f[-1:]])
               for f, g in zip(new, F)]
        return new, mix

    def step(self, X, dt, re, theta, keep=False):
        Z = X
        for s in range(3):
            if keep:
                def one(*a, s=s):
                    n = self.nf
                    x, z = self.stage(a[:n], a[n:2 * n], a[2 * n], a[2 * n + 1], a[2 * n + 2], s)
                    return (*x, *z)
                got = checkpoint(one, *X, *Z, dt, re, theta, use_reentrant=False)
                X, Z = list(got[:self.nf]), list(got[self.nf:])
            else:
                X, Z = self.stage(X, Z, dt, re, theta, s)
        return X

    def dense(self, X, nsteps):
        """The fields as a download returns them: periodic x/y ghosts on planes
        1..npz; the outer planes those of the start, the density inverted once
        a stage (mirrored first with density diffusion, over the whole plane)."""
        out = []
        for q, f in enumerate(X):
            full = self.full[q].clone()
            g = torch.cat([f[:, -1:], f, f[:, :1]], 1)
            g = torch.cat([g[:, :, -1:], g, g[:, :, :1]], 2)
            full[1:-1] = g[1:-1]
            if q == 3:
                for k in (0, -1):
                    if self.c.id:
                        full[k] = g[k]
                    else:
                        for _ in range(3 * nsteps):
                            full[k] = 1.0 / full[k]
            out.append(full)
        return out

    def march(self, nsteps):
        with torch.no_grad():
            X, t, dt = self.X, 0.0, None
            for _ in range(nsteps):
                dt = self.dt(X, self.re)
                t += float(dt)
                before = X
                X = self.step(X, dt, self.re, self.theta)
            _, mach = self.limits(before, self.re)
            return self.dense(X, nsteps), float(dt), t, float(torch.sqrt(mach.max()))

    def kinetic_energy(self, tt, re, theta, nsteps):
        X = list(self.X)
        X[4] = torch.cat([X[4][:1], tt, X[4][-1:]])
        for _ in range(nsteps):
            X = self.step(X, self.dt(X, re), re, theta, keep=True)
        ru, rv, rw, ro = (f[1:-1] for f in X[:4])
        vol = 1.0 / (self.x["dxxdx"] * self.y["dyydy"] * self.z["dzzdz"])
        return (vol * 0.5 * (ru * ru + rv * rv + rw * rw) / ro).sum()


def exact(c, seed):
    if c["physics"] == "relax" or cells_of(c) * c["steps"] > 1.5e9:
        return None  # the relaxation's planes are a chain of their own; the rest takes too long
    if c["kind"] == "ensemble":
        flat = []
        for f in member_flags(c, seed):
            fields, _, _, _ = Plain(pkg.Run(f)).march(c["steps"])
            flat += [q.reshape(-1).cpu() for q in fields]
        return torch.cat(flat)
    run_ = pkg.Run(flags(c, seed))
    p = Plain(run_)
    if c["kind"] == "adjoint":
        tt = perturbed(torch.from_numpy(np.array(run_.state(copy=False)["tt"][1:-1, 1:-1, 1:-1]))
                       .cuda(), seed).requires_grad_(True)
        p.re.requires_grad_(True)
        p.theta.requires_grad_(True)
        J = p.kinetic_energy(tt, p.re, p.theta, c["steps"])
        J.backward()
        return {"J": J.detach(), "tt": tt.grad, "re": p.re.grad, "theta": p.theta.grad}
    fields, dt, timt, umach = p.march(c["steps"])
    return {"fields": [f.cpu() for f in fields], "dt": dt, "timt": timt, "umach": umach}
