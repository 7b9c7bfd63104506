"""The work that the framework is used for, as cases that can be timed and checked.

Three ways in, each as a user's program calls it:

* ``grid``: the state lives in the program's own device tensors and is advanced with
  ``native.run_noalloc`` (hydro 2D/3D and 2D MHD);
* ``job``: one run from host memory to host memory with a ``native.Context`` that the program
  keeps: upload, steps, download (the way every 3D MHD run goes);
* ``batch``: many independent 2D blasts through a ``pool.Pool``: admit, step, download, retire.

Every initial state is a smooth random flow (a few Fourier modes in density, velocity, pressure
and, for MHD, a divergence-free field) with a strong blast in it, so that quiet, smooth and
shocked cells all occur. ``exact`` restates the schemes in plain float64 torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from euler_kokkos_amd import native, pool
from euler_kokkos_amd.params import make_params

REFLECT, OUTFLOW, PERIODIC = 1, 2, 3
BOUNDARIES = {"walls": REFLECT, "outflow": OUTFLOW, "periodic": PERIODIC}
SOLVER = {"hydro2d": "Hydro_Muscl_2D", "hydro3d": "Hydro_Muscl_3D", "mhd2d": "MHD_Muscl_2D", "mhd3d": "MHD_Muscl_3D"}
NVAR = {"hydro2d": 4, "hydro3d": 5, "mhd2d": 8, "mhd3d": 8}
# additions, multiplications, divisions, roots and comparisons of one cell and step
FLOPS = {"hydro2d": 345, "hydro3d": 580, "mhd2d": 1500, "mhd3d": 3200}
FOREVER = 1e30


def _case(name, via, path, shape, dtype, steps, riemann, bc, slope=2):
    nx, ny, nz = (tuple(shape) + (1,))[:3]
    c = dict(via=via, path=path, nx=nx, ny=ny, nz=nz, dtype=dtype, steps=steps, riemann=riemann, bc=bc, slope=slope)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a 64^2 grid with walls, where launches and their latency are all there is
        _case("hydro2d_64_f64", "grid", "hydro2d", (64, 64), "f64", 20, "hllc", "walls"),
        # the 512^2 implosion's grid, walls and solver (settings/implode_2D_512.ini)
        _case("hydro2d_512_f64", "grid", "hydro2d", (512, 512), "f64", 40, "hllc", "walls"),
        # a ragged 2D grid with the solver and slopes that a parameter file gets by default
        _case("hydro2d_1000x333_f32", "grid", "hydro2d", (1000, 333), "f32", 40, "approx", "outflow", 1),
        # an ordinary 3D run, no axis a multiple of a tile
        _case("hydro3d_101x75x130_f64", "grid", "hydro3d", (101, 75, 130), "f64", 20, "hllc", "outflow"),
        # the headline 3D blast (settings/blast_3D_256.ini), exact and bulk precision
        _case("hydro3d_256_f64", "grid", "hydro3d", (256, 256, 256), "f64", 10, "hllc", "periodic"),
        _case("hydro3d_256_f32", "grid", "hydro3d", (256, 256, 256), "f32", 10, "hllc", "periodic"),
        # a small ragged 2D MHD run between walls
        _case("mhd2d_300x211_f64", "grid", "mhd2d", (300, 211), "f64", 30, "hlld", "walls"),
        # the Orszag-Tang grid (settings/orszag_tang_2D_1024.ini), exact and bulk precision
        _case("mhd2d_1024_f64", "grid", "mhd2d", (1024, 1024), "f64", 10, "hlld", "periodic"),
        _case("mhd2d_1024_f32", "grid", "mhd2d", (1024, 1024), "f32", 20, "hlld", "periodic"),
        # the served 3D MHD blast: 50 steps from a host state to a host state
        _case("mhd3d_128_f64", "job", "mhd3d", (128, 128, 128), "f64", 50, "hlld", "periodic"),
        _case("mhd3d_97x64x110_f32", "job", "mhd3d", (97, 64, 110), "f32", 50, "hlld", "periodic"),
        # batched 2D blasts of mixed sizes, advanced together
        dict(name="batch2d_24_f32", via="batch", path="hydro2d", runs=24, edge=320, dtype="f32", steps=100,
             riemann="hllc", bc="walls", slope=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: any path, size, boundary and precision that they stand for."""
    kind = rng.choice(["hydro2d", "hydro3d", "mhd2d", "mhd3d", "batch"])
    dtype = rng.choice(["f64", "f32"])
    bc = rng.choice(sorted(BOUNDARIES))
    slope = rng.choice([1, 2, 2])
    if kind == "batch":
        return dict(via="batch", path="hydro2d", runs=rng.randint(6, 24), edge=rng.randint(64, 320), dtype=dtype,
                    steps=rng.randint(30, 100), riemann="hllc", bc="walls", slope=2)
    if kind == "hydro2d":
        return _case(None, "grid", kind, (_log(rng, 48, 1500), _log(rng, 48, 1200)), dtype, rng.randint(10, 40),
                     rng.choice(["hllc", "hllc", "approx"]), bc, slope)
    if kind == "hydro3d":
        shape = tuple(_log(rng, 24, 224) for _ in range(3))
        return _case(None, "grid", kind, shape, dtype, rng.randint(5, 10), rng.choice(["hllc", "hllc", "approx"]), bc, slope)
    if kind == "mhd2d":
        return _case(None, "grid", kind, (_log(rng, 40, 1024), _log(rng, 40, 1000)), dtype, rng.randint(5, 10), "hlld", bc, slope)
    shape = tuple(_log(rng, 20, 120) for _ in range(3))
    return _case(None, "job", kind, shape, dtype, rng.randint(20, 50), "hlld", bc, slope)


def _params(case, nx=None, ny=None, nz=None):
    mhd = case["path"].startswith("mhd")
    return make_params(SOLVER[case["path"]], nx or case["nx"], ny or case["ny"], nz or case.get("nz", 1),
                       gamma0="1.6666667" if mhd else "1.4", cfl="0.8" if mhd else "0.5",
                       slope_type=str(case["slope"]), riemann=case["riemann"], bc=(BOUNDARIES[case["bc"]],) * 6,
                       precision=native.EK_FP64 if case["dtype"] == "f64" else native.EK_FP32)


def _modes(rng, coords, amplitude, count=4):
    """A smooth periodic random field."""
    f = 0.0
    for _ in range(count):
        phase = sum(2 * math.pi * int(rng.integers(-3, 4)) * x for x in coords) + float(rng.uniform(0, 2 * math.pi))
        f = f + amplitude / math.sqrt(count) * float(rng.normal()) * torch.sin(phase)
    return f


def _initial(p, seed, index=0):
    """The conserved state U[var][k][j][i] in float64 on the GPU."""
    rng = np.random.default_rng([seed, index])
    n, d, lo = (p.nx, p.ny, p.nz), (p.dx, p.dy, p.dz), (p.xmin, p.ymin, p.zmin)

    def axes(shift):
        out = []
        for a in range(p.dim):
            x = lo[a] + (torch.arange(n[a], dtype=torch.float64, device="cuda") + shift[a]) * d[a]
            out.append(x.reshape([-1 if b == a else 1 for b in reversed(range(p.dim))]))
        return out

    at = axes((0.5, 0.5, 0.5))
    shape = tuple(reversed(n[:p.dim]))
    full = torch.zeros(shape, dtype=torch.float64, device="cuda")
    rho = 1.0 + 0.4 * torch.tanh(_modes(rng, at, 0.5) + full)
    vel = [_modes(rng, at, 0.4) + full for _ in range(3 if p.dim == 3 or p.mhd else 2)]
    r2 = sum((x - float(rng.uniform(0.2, 0.8))) ** 2 for x in at)
    press = 1.0 + 0.3 * torch.tanh(_modes(rng, at, 0.5) + full)
    press = torch.where(r2 < float(rng.uniform(0.08, 0.15)) ** 2, 10.0 ** float(rng.uniform(0.7, 1.5)) * press, press)
    U = torch.zeros((p.nbvar,) + shape, dtype=torch.float64, device="cuda")
    U[0] = rho
    for a, v in enumerate(vel):
        U[2 + a] = rho * v
    U[1] = press / (p.gamma0 - 1.0) + 0.5 * rho * sum(v * v for v in vel)
    if p.mhd:
        # in-plane field from a vector potential on the cell edges, so that its divergence is zero
        terms = [(int(rng.integers(-3, 4)), int(rng.integers(-3, 4)), float(rng.uniform(0, 2 * math.pi)),
                  0.05 * float(rng.normal())) for _ in range(4)]

        def potential(shift):
            x, y = axes(shift)[:2]
            return sum(c * torch.sin(2 * math.pi * (kx * x + ky * y) + f) for kx, ky, f, c in terms)

        a0 = potential((0, 0, 0))
        U[5] = float(rng.uniform(0.1, 0.5)) + (potential((0, 1, 0)) - a0) / p.dy
        U[6] = float(rng.uniform(0.1, 0.5)) - (potential((1, 0, 0)) - a0) / p.dx
        U[7] = float(rng.uniform(0.1, 0.5))
        right = [torch.roll(U[5], -1, -1), torch.roll(U[6], -1, -2)]
        U[1] += 0.125 * ((U[5] + right[0]) ** 2 + (U[6] + right[1]) ** 2) + 0.5 * U[7] ** 2
    return U


def _jobs(case, seed):
    """(params, state) of each run of a batch: square blasts, edges spread over 64..case["edge"]."""
    out = []
    for r in range(case["runs"]):
        n = 64 + int((case["edge"] - 64) * (0.381966 * (r + 1) % 1.0) + 0.5)
        p = _params(case, n, n, 1)
        out.append((p, _initial(p, seed, r)))
    return out


def prepare(case, seed):
    if case["via"] == "batch":
        jobs = [(p, U.cpu().numpy()) for p, U in _jobs(case, seed)]
        per = 8 if case["dtype"] == "f64" else 4
        room = sum(2 * 4 * p.nx * p.ny * per + 4096 for p, _ in jobs) + (64 << 20)
        return dict(case=case, jobs=jobs, pool=pool.Pool(jobs[0][0], room, len(jobs)))
    p = _params(case)
    U = _initial(p, seed)
    if case["via"] == "job":
        return dict(case=case, ctx=native.Context(p), host=native.pinned_copy(U.cpu().numpy()))
    U = U.to(torch.float64 if case["dtype"] == "f64" else torch.float32)
    return dict(case=case, params=p, start=U, U=torch.empty_like(U), U2=torch.empty_like(U))


def run(state):
    case = state["case"]
    steps = case["steps"]
    if case["via"] == "batch":
        P = state["pool"]
        ids = [P.admit(p, U, steps) for p, U in state["jobs"]]
        P.step(steps)
        out = [P.download(j) for j in ids]
        for j in ids:
            P.retire(j)
        return {"U": out}
    if case["via"] == "job":
        ctx = state["ctx"]
        ctx.upload(state["host"], native.EK_LAYOUT_SOA)
        t, it, dt = ctx.run(steps, steps, FOREVER)
        return {"U": ctx.download(native.EK_LAYOUT_SOA), "t": t, "it": it, "dt": dt}
    U, U2 = state["U"], state["U2"]
    U.copy_(state["start"])
    t, it, dt, second = native.run_noalloc(state["params"], U.data_ptr(), U2.data_ptr(), steps, steps, FOREVER,
                                           stream=torch.cuda.current_stream().cuda_stream)
    return {"U": U2 if second else U, "t": t, "it": it, "dt": dt}


def work(case):
    """Every step reads the state and writes it; nothing else has to move."""
    cells = case["runs"] * ((64 + case["edge"]) / 2) ** 2 if case["via"] == "batch" else case["nx"] * case["ny"] * case["nz"]
    per = 8 if case["dtype"] == "f64" else 4
    return {"bytes": 2.0 * per * NVAR[case["path"]] * cells * case["steps"], "flops": float(FLOPS[case["path"]]) * cells * case["steps"]}


# ------------------------------------------------------------------------------------------
# The schemes in float64. Arrays are [k][j][i] with ghost cells; axis 0 (x) is the last one.
# Neighbours come from torch.roll: what it wraps around reaches ghost cells only.


class _Scheme:
    def __init__(self, p):
        self.p, self.dim, self.mhd = p, p.dim, bool(p.mhd)
        self.g = 4 if self.mhd else 2
        self.d = (p.dx, p.dy, p.dz)[:p.dim]
        self.riemann = {0: self.approx, 3: self.hllc, 4: self.hlld}[p.riemann]

    def at(self, q, axis, off):
        """The value `off` cells further along `axis`."""
        return torch.roll(q, -off, dims=-1 - axis)

    def ghosts(self, U):
        """Ghost cells on each axis in turn; a wall turns the normal momentum (and normal field) round."""
        for a in range(self.dim):
            n, g = U.shape[-1 - a], self.g
            i = torch.arange(-g, n + g, device=U.device)
            kind = self.p.bc[2 * a]
            outside = (i < 0) | (i >= n)
            if kind == PERIODIC:
                src = i % n
            elif kind == OUTFLOW:
                src = i.clamp(0, n - 1)
            else:
                src = torch.where(i < 0, -1 - i, torch.where(i >= n, 2 * n - 1 - i, i)).clamp(0, n - 1)
            U = U.index_select(U.dim() - 1 - a, src)
            if kind == REFLECT:
                sign = torch.where(outside, -1.0, 1.0).to(U).reshape([-1] + [1] * a)
                U[2 + a] *= sign
                if self.mhd:
                    U[5 + a] *= sign
        return U

    def inside(self, U):
        for a in range(self.dim):
            U = U.narrow(U.dim() - 1 - a, self.g, U.shape[-1 - a] - 2 * self.g)
        return U

    def primitives(self, U):
        p = self.p
        d = U[0].clamp(min=p.smallr)
        nv = 3 if self.mhd else self.dim
        v = [U[2 + a] / d for a in range(nv)]
        e = U[1]
        B = []
        if self.mhd:
            # 2D: the missing neighbour along z counts as zero
            B = [0.5 * (U[5 + a] + (self.at(U[5 + a], a, 1) if a < self.dim else 0.0)) for a in range(3)]
            e = e - 0.5 * sum(b * b for b in B)
        e = e / d - 0.5 * sum(x * x for x in v)
        return [d, torch.maximum((p.gamma0 - 1.0) * d * e, d * p.smallp)] + v + B

    def fast(self, q, a):
        b2 = q[5] * q[5] + q[6] * q[6] + q[7] * q[7]
        c2 = self.p.gamma0 * q[1] / q[0]
        h = 0.5 * (b2 / q[0] + c2)
        return torch.sqrt(h + torch.sqrt(h * h - c2 * q[5 + a] * q[5 + a] / q[0]))

    def inv_dt(self, q):
        c = None if self.mhd else torch.sqrt(self.p.gamma0 * q[1] / q[0])
        s = sum(((self.fast(q, a) if self.mhd else c) + q[2 + a].abs()) / self.d[a] for a in range(self.dim))
        return float(self.inside(s[None]).max())

    def slope(self, q, axis):
        lo, hi = self.at(q, axis, -1), self.at(q, axis, 1)
        st = self.p.slope_type
        left, right, mid = st * (q - lo), st * (hi - q), 0.5 * (hi - lo)
        m = torch.minimum(torch.minimum(left.abs(), right.abs()), mid.abs())
        m = torch.where(left * right <= 0, 0.0, m)
        return torch.where(mid >= 0, m, -m)

    # -------------------------------------------------------------------------- hydro
    def hydro_step(self, U, q, dt):
        p, n = self.p, self.dim
        dq = [[self.slope(x, a) for x in q] for a in range(n)]
        div = sum(dq[a][2 + a] for a in range(n))

        def carried(v):
            return -sum(q[2 + a] * dq[a][v] for a in range(n))

        s = [carried(0) - div * q[0], carried(1) - div * p.gamma0 * q[1]]
        s += [carried(2 + a) - dq[a][1] / q[0] for a in range(n)]
        out = U.clone()
        for a in range(n):
            r = dt / self.d[a]
            lo = [q[v] - 0.5 * dq[a][v] + 0.5 * r * s[v] for v in range(n + 2)]
            hi = [q[v] + 0.5 * dq[a][v] + 0.5 * r * s[v] for v in range(n + 2)]
            lo[0], hi[0] = lo[0].clamp(min=p.smallr), hi[0].clamp(min=p.smallr)
            order = list(range(n + 2))
            order[2], order[2 + a] = order[2 + a], order[2]
            f = self.riemann([self.at(hi[v], a, -1) for v in order], [lo[v] for v in order])
            for v in range(n + 2):
                out[order[v]] += r * (f[v] - self.at(f[v], a, 1))
        return out

    def hllc(self, l, r):
        p = self.p
        side = []
        for q in (l, r):
            d = q[0].clamp(min=p.smallr)
            pr = torch.maximum(q[1], d * p.smallp)
            c = torch.sqrt((p.gamma0 * pr / d).clamp(min=p.smallc * p.smallc))
            side.append((d, pr, q[2], pr / (p.gamma0 - 1.0) + 0.5 * d * sum(x * x for x in q[2:]), c))
        (rl, pl, ul, el, cl), (rr, pr, ur, er, cr) = side
        c = torch.maximum(cl, cr)
        sl, sr = torch.minimum(ul, ur) - c, torch.maximum(ul, ur) + c
        rcl, rcr = rl * (ul - sl), rr * (sr - ur)
        us = (rcr * ur + rcl * ul + (pl - pr)) / (rcr + rcl)
        ps = (rcr * pl + rcl * pr + rcl * rcr * (ul - ur)) / (rcr + rcl)
        left = us > 0
        d, s, u, px, e = (torch.where(left, x, y) for x, y in ((rl, rr), (sl, sr), (ul, ur), (pl, pr), (el, er)))
        m = s - u
        star = (d * m / (s - us), us, ps, (m * e - px * u + ps * us) / (s - us))
        inner = left | (sr > 0)
        ro, uo, po, eo = (torch.where(sl > 0, x, torch.where(inner, y, z))
                          for x, y, z in zip((rl, ul, pl, el), star, (rr, ur, pr, er)))
        f = ro * uo
        return [f, (eo + po) * uo, f * uo + po] + [f * torch.where(f > 0, x, y) for x, y in zip(l[3:], r[3:])]

    def approx(self, l, r):
        p = self.p
        rl, rr = l[0].clamp(min=p.smallr), r[0].clamp(min=p.smallr)
        pl, pr = torch.maximum(l[1], rl * p.smallp), torch.maximum(r[1], rr * p.smallp)
        ul, ur = l[2], r[2]
        cl, cr = p.gamma0 * pl * rl, p.gamma0 * pr * rr

        def mass(c, ref, x):
            return torch.sqrt(c * (1.0 + p.gamma6 * (x - ref) / ref))

        wl, wr = torch.sqrt(cl), torch.sqrt(cr)
        x = (((wr * pl + wl * pr) + wl * wr * (ul - ur)) / (wl + wr)).clamp(min=0.0)
        active = torch.ones_like(x, dtype=torch.bool)
        for _ in range(10):
            a, b = mass(cl, pl, x), mass(cr, pr, x)
            ql, qr = 2 * a ** 3 / (a * a + cl), 2 * b ** 3 / (b * b + cr)
            step = torch.maximum(qr * ql / (qr + ql) * ((ul - (x - pl) / a) - (ur + (x - pr) / b)), -x)
            x = torch.where(active, x + step, x)
            active = active & ((step / (x + p.smallpp)).abs() > 1e-6)
        wl, wr = mass(cl, pl, x), mass(cr, pr, x)
        us = 0.5 * (ul + (pl - x) / wl + ur - (pr - x) / wr)
        left = torch.copysign(torch.ones_like(us), us) > 0
        sgn = torch.where(left, 1.0, -1.0)
        ro, uo, po, wo = (torch.where(left, y, z) for y, z in ((rl, rr), (ul, ur), (pl, pr), (wl, wr)))
        co = torch.sqrt((p.gamma0 * po / ro).abs()).clamp(min=p.smallc)
        rs = (ro / (1.0 + ro * (po - x) / (wo * wo))).clamp(min=p.smallr)
        cs = torch.sqrt((p.gamma0 * x / rs).abs()).clamp(min=p.smallc)
        shock = wo / ro - sgn * uo
        hit = x >= po
        out, into = torch.where(hit, shock, co - sgn * uo), torch.where(hit, shock, cs - sgn * us)
        frac = 0.5 * (1.0 + (out + into) / torch.maximum(out - into, p.smallc + (out + into).abs()))
        frac = torch.nan_to_num(frac, nan=0.0).clamp(0.0, 1.0)
        d, u, pg = (frac * y + (1.0 - frac) * z for y, z in ((rs, ro), (us, uo), (x, po)))
        d, u, pg = (torch.where(into > 0, y, torch.where(out < 0, z, m))
                    for y, z, m in ((rs, ro, d), (us, uo, u), (x, po, pg)))
        rest = [torch.where(left, y, z) for y, z in zip(l[3:], r[3:])]
        f = d * u
        e = pg / (p.gamma0 - 1.0) + 0.5 * d * (u * u + sum(y * y for y in rest))
        return [f, u * (e + pg), f * u + pg] + [f * y for y in rest]

    # ---------------------------------------------------------------------------- MHD
    def floors(self, q):
        q[0] = q[0].clamp(min=self.p.smallr)
        q[1] = torch.maximum(q[1], self.p.smallp * (q[0] if self.dim == 2 else torch.ones_like(q[0])))
        return q

    def mhd_step(self, U, q, dt):
        p, n = self.p, self.dim
        ratio = [dt / x for x in self.d]
        edges = (2,) if n == 2 else (0, 1, 2)
        dq = [[0.5 * self.slope(x, a) for x in q] for a in range(n)]
        face = [U[5], U[6], U[7]]
        # transverse half slopes of the face fields and the edge fields v x B before the step
        dface = {(m, a): 0.5 * self.slope(face[m], a) for m in range(n) for a in range(n) if a != m}
        E = {}
        for k in edges:
            i, j = (k + 1) % 3, (k + 2) % 3

            def corner(x):
                y = x + self.at(x, i, -1)
                return 0.25 * (y + self.at(y, j, -1))

            E[k] = (corner(q[2 + i]) * 0.5 * (face[j] + self.at(face[j], i, -1))
                    - corner(q[2 + j]) * 0.5 * (face[i] + self.at(face[i], j, -1)))
        left = [f.clone() for f in face]
        for i in range(n):
            j, k = (i + 1) % 3, (i + 2) % 3
            if k in E:
                left[i] = left[i] + 0.5 * (self.at(E[k], j, 1) - E[k]) * ratio[j]
            if j in E:
                left[i] = left[i] - 0.5 * (self.at(E[j], k, 1) - E[j]) * ratio[k]
        right = [self.at(left[i], i, 1) for i in range(n)]
        dnormal = [0.5 * (self.at(face[i], i, 1) - face[i]) for i in range(n)]
        r, pr, v, B = q[0], q[1], q[2:5], q[5:8]
        c = [x.clone() for x in q]
        for a in range(n):
            t, g = ratio[a], dq[a]
            c[0] = c[0] + (-v[a] * g[0] - g[2 + a] * r) * t
            c[1] = c[1] + (-v[a] * g[1] - g[2 + a] * p.gamma0 * pr) * t
            across = sum(B[m] * g[5 + m] for m in range(3) if m != a)
            for i in range(3):
                force = -(g[1] + across) / r if i == a else B[a] * g[5 + i] / r
                c[2 + i] = c[2 + i] + (-v[a] * g[2 + i] + force) * t
                if i != a:
                    c[5 + i] = c[5 + i] + (v[i] * dnormal[a] + B[a] * g[2 + i] - v[a] * g[5 + i] - B[i] * g[2 + a]) * t
        out = U.clone()
        for a in range(n):
            hi = self.floors([x + y for x, y in zip(c, dq[a])])
            lo = self.floors([x - y for x, y in zip(c, dq[a])])
            hi[5 + a], lo[5 + a] = right[a], left[a]
            order = list(range(8))
            order[2], order[2 + a] = order[2 + a], order[2]
            order[5], order[5 + a] = order[5 + a], order[5]
            f = self.riemann([self.at(hi[m], a, -1) for m in order], [lo[m] for m in order])
            for m in range(8):
                to = order[m]
                if to < 5 or (to == 7 and n == 2):
                    out[to] += ratio[a] * (f[m] - self.at(f[m], a, 1))
        F = {}
        for k in edges:
            i, j = (k + 1) % 3, (k + 2) % 3

            def state(hi_i, hi_j):
                s = [x + (y if hi_i else -y) + (z if hi_j else -z) for x, y, z in zip(c, dq[i], dq[j])]
                s = self.floors(s)
                bi, bj = (right if hi_i else left)[i], (right if hi_j else left)[j]
                di, dj = dface[i, j], dface[j, i]
                di, dj = (self.at(di, i, 1) if hi_i else di), (self.at(dj, j, 1) if hi_j else dj)
                s = [s[0], s[1], s[2 + i], s[2 + j], bi + (di if hi_j else -di), bj + (dj if hi_i else -dj), s[5 + k]]
                if hi_i:
                    s = [self.at(x, i, -1) for x in s]
                return [self.at(x, j, -1) for x in s] if hi_j else s

            F[k] = self.emf(state(True, True), state(True, False), state(False, True), state(False, False))
        for i in range(n):
            j, k = (i + 1) % 3, (i + 2) % 3
            if k in F:
                out[5 + i] += (self.at(F[k], j, 1) - F[k]) * ratio[j]
            if j in F:
                out[5 + i] -= (self.at(F[j], k, 1) - F[j]) * ratio[k]
        return out

    def hlld(self, l, r):
        p = self.p
        a = 0.5 * (l[5] + r[5])
        sgn = torch.where(a >= 0, 1.0, -1.0)
        side = []
        for q in (l, r):
            mag = 0.5 * (a * a + q[6] * q[6] + q[7] * q[7])
            e = q[1] / (p.gamma0 - 1.0) + 0.5 * (q[2] * q[2] + q[3] * q[3] + q[4] * q[4]) * q[0] + mag
            side.append((q[0], q[2], q[3], q[4], q[6], q[7], q[1] + mag, e, q[2] * a + q[3] * q[6] + q[4] * q[7],
                         self.fast(q[:5] + [a] + q[6:], 0)))
        (rl, ul, _, _, _, _, ptl, _, _, cl), (rr, ur, _, _, _, _, ptr, _, _, cr) = side
        c = torch.maximum(cl, cr)
        sl, sr = torch.minimum(ul, ur) - c, torch.maximum(ul, ur) + c
        rcl, rcr = rl * (ul - sl), rr * (sr - ur)
        us = (rcr * ur + rcl * ul + (ptl - ptr)) / (rcr + rcl)
        pts = (rcr * ptl + rcl * ptr + rcl * rcr * (ul - ur)) / (rcr + rcl)
        stars = []
        for s, (d, u, v, w, b, cc, pt, e, vb, _) in zip((sl, sr), side):
            ds = d * (s - u) / (s - us)
            es, ef = d * (s - u) * (s - us) - a * a, d * (s - u) * (s - u) - a * a
            same = (a * a > 0) & ((es / (a * a) - 1.0).abs() <= 1e-8)
            vs, ws = torch.where(same, v, v - a * b * (us - u) / es), torch.where(same, w, w - a * cc * (us - u) / es)
            bs, cs = torch.where(same, b, b * ef / es), torch.where(same, cc, cc * ef / es)
            vbs = us * a + vs * bs + ws * cs
            ets = ((s - u) * e - pt * u + pts * us + a * (vb - vbs)) / (s - us)
            stars.append((ds, us, vs, ws, bs, cs, pts, ets, vbs))
        (dl, _, vl, wl, bl, ccl, _, etl, vbl), (dr, _, vr, wr, br, ccr, _, etr, vbr) = stars
        ql, qr = torch.sqrt(dl), torch.sqrt(dr)
        den = ql + qr
        vs, ws = (ql * vl + qr * vr + sgn * (br - bl)) / den, (ql * wl + qr * wr + sgn * (ccr - ccl)) / den
        bs = (ql * br + qr * bl + sgn * ql * qr * (vr - vl)) / den
        cs = (ql * ccr + qr * ccl + sgn * ql * qr * (wr - wl)) / den
        vb = us * a + vs * bs + ws * cs
        twol = (dl, us, vs, ws, bs, cs, pts, etl - sgn * ql * (vbl - vb), vb)
        twor = (dr, us, vs, ws, bs, cs, pts, etr + sgn * qr * (vbr - vb), vb)
        out = side[1]
        for cond, value in ((sr > 0, stars[1]), (us + a.abs() / qr > 0, twor), (us > 0, twol),
                            (us - a.abs() / ql > 0, stars[0]), (sl > 0, side[0])):
            out = [torch.where(cond, x, y) for x, y in zip(value, out)]
        d, u, v, w, b, cc, pt, e, vb = out[:9]
        return [d * u, (e + pt) * u - a * vb, d * u * u - a * a + pt, d * u * v - a * b, d * u * w - a * cc,
                torch.zeros_like(a), b * u - a * v, cc * u - a * w]

    def emf(self, s00, s01, s10, s11):
        """The edge field from the four states around an edge; s01: low along the first axis, high along the
        second. A state is r, p, u, v, a, b, c."""
        S = {(0, 0): list(s00), (0, 1): list(s01), (1, 0): list(s10), (1, 1): list(s11)}
        for j in (0, 1):
            m = 0.5 * (S[0, j][4] + S[1, j][4])
            S[0, j][4] = S[1, j][4] = m
        for i in (0, 1):
            m = 0.5 * (S[i, 0][5] + S[i, 1][5])
            S[i, 0][5] = S[i, 1][5] = m
        keys = list(S)

        def most(f):
            x = f(*keys[0])
            for k in keys[1:]:
                x = torch.maximum(x, f(*k))
            return x

        def fast(i, j, axis):
            r, pr, _, _, a, b, c = S[i, j]
            return self.fast([r, pr, None, None, None, a, b, c], axis)

        u, v = (lambda i, j: S[i, j][2]), (lambda i, j: S[i, j][3])
        fx, fy = most(lambda i, j: fast(i, j, 0)), most(lambda i, j: fast(i, j, 1))
        s = [-most(lambda i, j: -u(i, j)) - fx, most(u) + fx]
        t = [-most(lambda i, j: -v(i, j)) - fy, most(v) + fy]
        pt = {k: x[1] + 0.5 * (x[4] ** 2 + x[5] ** 2 + x[6] ** 2) for k, x in S.items()}
        mx = {(i, j): S[i, j][0] * ((u(i, j) - s[0]) if i == 0 else (s[1] - u(i, j))) for i, j in keys}
        my = {(i, j): S[i, j][0] * ((v(i, j) - t[0]) if j == 0 else (t[1] - v(i, j))) for i, j in keys}
        us = (sum(mx[k] * u(*k) for k in keys) + pt[0, 0] + pt[0, 1] - pt[1, 0] - pt[1, 1]) / sum(mx.values())
        vs = (sum(my[k] * v(*k) for k in keys) + pt[0, 0] + pt[1, 0] - pt[0, 1] - pt[1, 1]) / sum(my.values())
        A, Bs, ex, ey, e, plain = {}, {}, {}, {}, {}, {}
        alf = {"L": [], "R": [], "B": [], "T": []}
        for i, j in keys:
            r, _, uu, vv, a, b, _ = S[i, j]
            kx, ky = (s[i] - uu) / (s[i] - us), (t[j] - vv) / (t[j] - vs)
            Bs[i, j], A[i, j] = b * kx, a * ky
            plain[i, j], ex[i, j] = uu * b - vv * a, us * Bs[i, j] - vv * a
            ey[i, j], e[i, j] = uu * b - vs * A[i, j], us * Bs[i, j] - vs * A[i, j]
            rx, ry, rs = torch.sqrt(r * kx), torch.sqrt(r * ky), torch.sqrt(r * kx * ky)
            alf["LR"[i]] += [a.abs() / rx, A[i, j].abs() / rs]
            alf["BT"[j]] += [b.abs() / ry, Bs[i, j].abs() / rs]
        alf = {k: torch.stack(x).amax(0).clamp(min=self.p.smallc) for k, x in alf.items()}
        sal, sar = (us - alf["L"]).clamp(max=0.0), (us + alf["R"]).clamp(min=0.0)
        sab, sat = (vs - alf["B"]).clamp(max=0.0), (vs + alf["T"]).clamp(min=0.0)
        w, h = sar - sal, sat - sab
        at, ab = (sar * A[1, 1] - sal * A[0, 1]) / w, (sar * A[1, 0] - sal * A[0, 0]) / w
        br, bl = (sat * Bs[1, 1] - sab * Bs[1, 0]) / h, (sat * Bs[0, 1] - sab * Bs[0, 0]) / h
        middle = ((sal * sab * e[1, 1] - sal * sat * e[1, 0] - sar * sab * e[0, 1] + sar * sat * e[0, 0]) / w / h
                  - sat * sab / h * (at - ab) + sar * sal / w * (br - bl))

        def rowx(j):
            x = (sar * ex[0, j] - sal * ex[1, j] + sar * sal * (S[1, j][5] - S[0, j][5])) / w
            return torch.where(s[0] >= 0, plain[0, j], torch.where(s[1] < 0, plain[1, j], x))

        def coly(i):
            return (sat * ey[i, 0] - sab * ey[i, 1] - sat * sab * (S[i, 1][4] - S[i, 0][4])) / h

        x = torch.where(s[0] >= 0, coly(0), torch.where(s[1] < 0, coly(1), middle))
        return torch.where(t[0] >= 0, rowx(0), torch.where(t[1] < 0, rowx(1), x))

    def advance(self, U, steps):
        t = dt = 0.0
        for _ in range(steps):
            P = self.ghosts(U)
            q = self.primitives(P)
            dt = self.p.cfl / self.inv_dt(q)
            P = self.mhd_step(P, q, dt) if self.mhd else self.hydro_step(P, q, dt)
            U = self.inside(P).contiguous()
            t += dt
        return U, t, dt


def exact(case, seed):
    if case["via"] == "batch":
        return {"U": [_Scheme(p).advance(U, case["steps"])[0].cpu().numpy() for p, U in _jobs(case, seed)]}
    p = _params(case)
    U = _initial(p, seed)
    if case["via"] == "grid" and case["dtype"] == "f32":
        U = U.float().double()
    U, t, dt = _Scheme(p).advance(U, case["steps"])
    return {"U": U.cpu().numpy() if case["via"] == "job" else U, "t": t, "it": case["steps"], "dt": dt}
