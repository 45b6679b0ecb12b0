"""Timed workloads of the framework: what its users have it do, through the
public entry points of vlasolve_amd, over the sizes and options it takes.

A run of the solver advances f with a statistics line every 25 steps and a
snapshot of f at the end of a pass (the parameter defaults write statistics
every 25 steps and a snapshot every 500).  A gradient records a run and
sweeps it back (vls_record, vls_adjoint), from the same f0 and delay-line
values each time, as an optimiser's iteration does.  The profile call takes f
on the device and returns density, potential and enclosed mass there.

`exact` computes the same outputs with plain torch in float64: its own grid,
generators, feet and delay lines, dense inverses for the splines, gathers for
the evaluations and torch.autograd for the gradients.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import vlasolve_amd as V

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
STATS_EVERY = 25

# ------------------------------------------------------------------ the cases


def _case(name, kind, init, grids, steps, **more):
    c = {"name": name, "kind": kind, "init": init, "grids": grids, "steps": steps, "dt": 0.005,
         "species": 1, "no_linking": False, "kernel": "delayed", "buffer": 0, "every": 0}
    c.update(more)
    return c


def listed():
    """grids: cells of each run as r x v x j (r and v have one node more)."""
    return [
        # the smallest call: density, potential and enclosed mass of an f on the
        # device, as code under graph capture or in a tight loop asks for them
        _case("profile_65", "profile", "UDF", "64x64x32", 1),
        # the small headline configuration, 65 x 65 x 32: launches and latency count
        _case("run_udf_65", "run", "UDF", "64x64x32", 500),
        # the Hernquist generator's own default grid, 91 x 81 x 80: sizes that no
        # table of the solver lists
        _case("run_hernquist_91", "run", "Hernquist", "90x80x80", 500, dt=0.025),
        # the Plummer generator's own default grid, 181 x 81 x 80: long rows, short columns
        _case("run_plummer_181", "run", "Plummer", "180x80x80", 300, dt=0.1),
        # the option without linking (half drift, kick, half drift), reflective centre
        _case("run_nolinking_129", "run", "PLDF", "128x128x64", 250, no_linking=True,
              kernel="reflective"),
        # two species with delay lines and a buffer of two nodes around the centre
        _case("run_species_97", "run", "UDF", "96x96x48", 200, species=2, buffer=2),
        # the default grid of the uniform sphere, 201 x 201 x 200
        _case("run_udf_201", "run", "UDF", "200x200x200", 500),
        # the large configuration, 513 x 513 x 256
        _case("run_hernquist_513", "run", "Hernquist", "512x512x256", 100, dt=0.0025),
        # an ensemble of uneven runs stepped together
        _case("ensemble_8", "ensemble", "UDF",
              "64x64x64,96x128x64,128x64x96,192x96x64,256x128x128,64x192x128,128x256x96,192x192x128",
              150),
        # the gradient of a mass-profile loss, 129 x 129 x 64, checkpoints every 50 steps
        _case("gradient_129", "gradient", "PLDF", "128x128x64", 200, every=50),
        # the same on the default grid, every step kept
        _case("gradient_201", "gradient", "UDF", "200x200x200", 25, every=5),
        # gradients of a batch of uneven runs
        _case("gradient_batch_4", "batch", "Hernquist", "150x131x96,210x180x64,131x257x70,96x64x48",
              28, every=14, dt=0.0025),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, sizes spread over their logarithm, odd ones among them."""
    kind = rng.choice(["profile", "run", "run", "run", "ensemble", "gradient", "gradient", "batch"])
    init = rng.choice(["UDF", "PLDF", "Hernquist", "Plummer"])
    more = {"dt": rng.choice([0.0025, 0.005])}
    n_runs = {"ensemble": rng.randint(2, 6), "batch": rng.randint(2, 4)}.get(kind, 1)
    top = {"profile": 200, "run": 320, "ensemble": 200, "gradient": 220, "batch": 180}[kind]
    common = [64, 96, 128, 192, 200, 256]  # cell counts that users type
    grids, pts = [], 0
    for _ in range(n_runs):
        axis = [rng.choice([s for s in common if s <= top]) if rng.random() < 0.4 else _size(rng, 24, top)
                for _ in range(2)]
        axis.append(_size(rng, 12, min(top, 200)))
        grids.append("%dx%dx%d" % tuple(axis))
        pts += (axis[0] + 1) * (axis[1] + 1) * axis[2]
    if kind == "run":
        steps = max(25, min(300, int(8e8 / pts)))
        if init in ("UDF", "PLDF"):
            more["species"] = rng.choice([1, 1, 1, 2])
        more["no_linking"] = rng.random() < 0.25
        more["kernel"] = rng.choice(["delayed", "delayed", "reflective"])
        more["buffer"] = rng.choice([0, 0, 2]) if more["kernel"] == "delayed" else 0
    elif kind == "ensemble":
        steps = max(25, min(150, int(4e8 / pts)))
    else:
        steps = max(10, min(100, int(1e8 / pts)))
    if kind in ("gradient", "batch"):
        more["every"] = max(5, min(50, int(round(math.sqrt(steps)))))
    c = _case("", kind, init, ",".join(grids), 1 if kind == "profile" else steps, **more)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs


def _grids(case):
    return [tuple(int(x) for x in g.split("x")) for g in case["grids"].split(",")]


def _configs(case, seed):
    """Command-line style parameters of each run: the physical parameters come from the seed."""
    rng = random.Random(int(seed) * 7919 + 1)
    out = []
    for pr, pu, pj in _grids(case):
        init, nS = case["init"], case["species"]
        cfg = {"init.type": init, "grid.Pres": pr, "grid.Ures": [pu, pj], "solver.G": 1,
               "solver.dt": case["dt"], "solver.noLinking": int(case["no_linking"]),
               "solver.kernelType": case["kernel"], "solver.kernelBufferSize": case["buffer"],
               "solver.nSpecies": nS}
        if init == "UDF":
            cfg.update({"init.M": [1.0 / (k + 1) for k in range(nS)], "init.smoothingRadius": [0.5] * nS,
                        "init.alpha": [rng.uniform(0.1, 1.0) for _ in range(nS)],
                        "init.R0": [rng.uniform(1.5, 3.0) for _ in range(nS)],
                        "grid.Pmin": 0.01, "grid.Pmax": 25, "grid.Umin": [-2, 0],
                        "grid.Umax": [2, 1.6]})
        elif init == "PLDF":
            cfg.update({"init.M": [1.0 / (k + 1) for k in range(nS)], "init.smoothingRadius": [0.5] * nS,
                        "init.n": [1] * nS, "init.alpha": [1] * nS,
                        "init.eta": [rng.uniform(0.08, 0.15) for _ in range(nS)],
                        "grid.Pmin": 0.01, "grid.Pmax": 30, "grid.Umin": [-1.5, 0],
                        "grid.Umax": [1.5, 1.6]})
        elif init == "Hernquist":
            cfg.update({"init.M": rng.uniform(0.8, 1.0), "init.R0": rng.uniform(1.0, 1.4),
                        "grid.Pmin": 0.01, "grid.Pmax": 250, "grid.Umin": [-1.45, 1e-4],
                        "grid.Umax": [1.45, 12.96]})
        else:
            cfg.update({"init.M": rng.uniform(0.8, 1.0), "init.R0": rng.uniform(1.0, 1.4),
                        "grid.Pmin": 0.01, "grid.Pmax": 100, "grid.Umin": [-1.45, 0],
                        "grid.Umax": [1.45, 3.24]})
        out.append(cfg)
    return out


_stream = []


def _shared_stream():
    """One stream for every profile call: they share the device's scratch array."""
    if not _stream:
        _stream.append(torch.cuda.Stream())
    return _stream[0]


def prepare(case, seed):
    cfgs = _configs(case, seed)
    kind = case["kind"]
    st = {"kind": kind, "steps": case["steps"], "every": case["every"]}
    if kind in ("ensemble", "batch"):
        st["solver"] = V.Ensemble(cfgs)
        st["n"] = len(cfgs)
    else:
        st["solver"] = V.Solver(cfgs[0])
        st["n"] = 1
    if kind == "profile":
        s = st["solver"]
        st["ctx"] = s.context
        st["f"] = torch.from_numpy(s.f()).to(DEV)
        st["out"] = [torch.empty(s.nR, dtype=F64, device=DEV) for _ in range(3)]
        torch.cuda.synchronize()
        _shared_stream()
    if kind in ("gradient", "batch"):
        ctx = st["solver"].context
        st["f0"] = [ctx.download_f(k, tuple(ctx.info(k)[a] for a in ("nJ", "nU", "nR")))
                    for k in range(st["n"])]
        st["lines"] = [ctx.get_chains(k) for k in range(st["n"])]
        st["target"] = [ctx.mass_profile(k) for k in range(st["n"])]
    return st


def run(state):
    kind, s, n = state["kind"], state["solver"], state["n"]
    if kind == "profile":
        rho, phi, mass = state["out"]
        state["ctx"].density_potential_noalloc(state["f"].data_ptr(), rho.data_ptr(), phi.data_ptr(),
                                               mass.data_ptr(), stream=_shared_stream().cuda_stream)
        return {"rho": rho, "phi": phi, "mass": mass}
    if kind == "run":
        lines, left = [], state["steps"]
        while left > 0:
            s.step(min(STATS_EVERY, left))
            left -= STATS_EVERY
            lines.append(list(s.stats().values()))
        dM, acc, total = s.moments()
        return {"f": s.f(), "stats": np.array(lines), "dM": dM, "acc": acc, "total": total}
    ctx = s.context
    if kind == "ensemble":
        lines, left = [], state["steps"]
        while left > 0:
            s.step(min(STATS_EVERY, left))
            left -= STATS_EVERY
            lines.append([list(ctx.stats(k).values()) for k in range(n)])
        return {"f": [s.f(k) for k in range(n)], "stats": np.array(lines)}
    for k in range(n):
        ctx.upload_f(k, state["f0"][k])
        ctx.put_chains(*state["lines"][k], run=k)
    if kind == "gradient":
        ctx.record(state["steps"], state["every"])
    else:
        ctx.record_batch(state["steps"], state["every"])
    M = [ctx.mass_profile(k) for k in range(n)]
    dL = [2.0 * (M[k] - state["target"][k]) for k in range(n)]
    grads = [ctx.adjoint(dL_dM=dL[0])] if kind == "gradient" else ctx.adjoint_batch(dL_dM=dL)
    return {"mass": M, "grad_f0": [g[0] for g in grads], "grad_vals0": [g[1] for g in grads]}


def work(case):
    """Per step and point: f read and written (16 bytes a species), the foot of the
    drift read (16 bytes; twice without linking).  A gradient's reverse step reads
    the same again with the adjoint in place of f, and the kept acceleration only.
    A profile reads f once."""
    byt = flo = 0.0
    for pr, pu, pj in _grids(case):
        pts = (pr + 1) * (pu + 1) * pj
        if case["kind"] == "profile":
            byt += 8.0 * pts + 24 * (pr + 1)
            flo += 6.0 * pts
            continue
        drifts = 2 if case["no_linking"] else 1
        step_b = pts * (16.0 * case["species"] + 16.0 * drifts)
        step_f = pts * case["species"] * (6 + 24 + 25 + drifts * (2 * 24 + 60))
        times = case["steps"] * (2 if case["kind"] in ("gradient", "batch") else 1)
        byt += step_b * times + 8.0 * pts * case["species"]
        flo += step_f * times
    return {"bytes": byt, "flops": flo}


# ------------------------------------------------------------------ the same in plain torch, float64


def _t(x):
    return torch.as_tensor(np.asarray(x, dtype=np.float64), device=DEV)


def _axis(lo, hi, n, scale):
    if scale == "log":
        v = np.exp(np.linspace(math.log(lo), math.log(hi), n + 1))
    elif scale == "quad":
        v = np.linspace(math.sqrt(lo), math.sqrt(hi), n + 1) ** 2
    else:
        v = np.linspace(lo, hi, n + 1)
    v[0], v[-1] = lo, hi
    return v


class _Model:
    """One run: grid, initial f, feet, delay lines and the step."""

    def __init__(self, cfg):
        get = cfg.get
        self.dt, self.nS = get("solver.dt"), get("solver.nSpecies")
        self.linking = not get("solver.noLinking")
        self.R = _t(_axis(get("grid.Pmin"), get("grid.Pmax"), get("grid.Pres"), "log"))
        self.U = _t(_axis(get("grid.Umin")[0], get("grid.Umax")[0], get("grid.Ures")[0], "lin"))
        jscale = "log" if get("init.type") == "Hernquist" else "quad"
        # the cell value of a quadratic or logarithmic axis is the mean of its edges
        edges = _t(_axis(get("grid.Umin")[1], get("grid.Umax")[1], get("grid.Ures")[1], jscale))
        self.J = 0.5 * (edges[1:] + edges[:-1])
        self.nR, self.nU, self.nJ = len(self.R), len(self.U), len(self.J)
        self.dR = self.R[1:] - self.R[:-1]
        self.dU = self.U[1:] - self.U[:-1]
        dJ = edges[1:] - edges[:-1]
        dJ[self.nU - 1:] = 0.0  # the reference's widths stop at the number of v cells
        self.weight = 8 * math.pi ** 2 * self.J * dJ
        self.hr = (self.nR - 1) / float(torch.log(self.R[-1] / self.R[0]))
        self.hu = (self.nU - 1) / float(self.U[-1] - self.U[0])
        self.invR, self.invU = self._spline(self.nR), self._spline(self.nU)
        r, u, j = self.R[None, None, :], self.U[None, :, None], self.J[:, None, None]
        self.f = [self._value(cfg, s, r, u, j).expand(self.nJ, self.nU, self.nR).clone()
                  for s in range(self.nS)]
        dth = self.dt if self.linking else 0.5 * self.dt
        kr = float(self.R[get("solver.kernelBufferSize")])
        delayed = get("solver.kernelType") == "delayed"
        ru = [a.expand(self.nJ, self.nU, self.nR).reshape(-1) for a in (r, u, j)]
        fr, fu = self._foot(*ru, dth, -1.0 if delayed else kr)
        inner = (fr < kr) if delayed else torch.zeros_like(fr, dtype=torch.bool)
        gone = (fr >= self.R[-1]) | (fr <= self.R[0]) | (fu >= self.U[-1]) | (fu <= self.U[0])
        self.live = ~(inner | gone)
        self.foot = self._stencil(fr, fu, self.live)
        # delay lines: where the orbit was at earlier multiples of the drift's step
        self.point = torch.nonzero(inner).reshape(-1)
        nc = len(self.point)
        pr, pu, pj = (a[self.point] for a in ru)
        self.len = torch.zeros(nc, dtype=torch.int64, device=DEV)
        parts, active, k = [], torch.arange(nc, device=DEV), 1
        while len(active):
            cr, cu = self._foot(pr[active], pu[active], pj[active], k * dth, -1.0)
            val = torch.stack([self._value(cfg, s, cr, cu, pj[active]) for s in range(self.nS)])
            stay = cr < kr
            parts.append((active, torch.where(stay, val, torch.zeros_like(val)), cr, cu))
            self.len[active] += 1
            active = active[stay]
            k += 1
        self.off = torch.cumsum(self.len, 0) - self.len
        cells = int(self.len.sum())
        self.vals = [torch.zeros(cells, dtype=F64, device=DEV) for _ in range(self.nS)]
        br, bu = torch.zeros_like(pr), torch.zeros_like(pr)
        for k, (at, val, cr, cu) in enumerate(parts):
            for s in range(self.nS):
                self.vals[s][self.off[at] + k] = val[s]
            br[at], bu[at] = cr, cu  # the last written is the back cell
        self.head = torch.zeros_like(self.len)
        back_in = (bu > self.U[0]) & (bu < self.U[-1])
        self.back_in = back_in
        self.back = self._stencil(br, bu, back_in, self.point)
        for s in range(self.nS):  # renormalised to the species' mass
            mass = get("init.M")
            mass = mass[s] if isinstance(mass, list) else mass
            fac = mass / float(self._moment(self.f[s]).sum())
            self.f[s] = self.f[s] * fac
            self.vals[s] = self.vals[s] * fac

    @staticmethod
    def _spline(n):
        """Inverse of the natural cubic B-spline system: n values to n + 2 coefficients."""
        A = np.zeros((n + 2, n + 2))
        A[0, :3] = A[-1, -3:] = (1, -2, 1)
        for k in range(1, n + 1):
            A[k, k - 1:k + 2] = (1 / 6, 4 / 6, 1 / 6)
        return _t(np.linalg.inv(A)[:, 1:-1])

    @staticmethod
    def _value(cfg, s, r, u, j):
        """The distribution functions of the four generators."""
        def p(key):
            v = cfg["init." + key]
            return v[s] if isinstance(v, list) else v
        kind, M = cfg["init.type"], p("M")
        if kind == "UDF":
            R0, s2 = p("R0"), p("alpha") / (5 * p("R0"))
            rho = 3 * M / (4 * math.pi * R0 ** 3)
            edge = 0.5 * (1 + torch.erf((R0 - r) / p("smoothingRadius")))
            f = edge * rho * (2 * math.pi * s2) ** -1.5 * torch.exp(-(u * u + (j / r) ** 2) / (2 * s2))
            return torch.clamp(f, min=1e-200)
        if kind == "PLDF":
            n, eta, alpha = p("n"), p("eta"), p("alpha")
            R0 = 1 / eta
            rho = (3 - n) * M / (4 * math.pi * R0 ** (3 - n))
            so = (3 - n) / (5 - 2 * n) * (M * eta) / (R0 * (alpha * 0.5 + 1))
            sr = so * 0.5 * alpha
            edge = 0.5 * (1 + torch.erf((R0 - r) / p("smoothingRadius")))
            f = edge * rho / (math.sqrt(2 * sr * math.pi ** 3) * so) * r ** -n * \
                torch.exp(-u * u / (2 * sr) - (j / r) ** 2 / so)
            return torch.clamp(f, min=1e-200)
        R0 = p("R0")
        kin = 0.5 * (u * u + (j / r) ** 2)
        if kind == "Plummer":
            eps = kin - M / torch.sqrt(r * r + R0 * R0)
            bound = torch.clamp(-eps, min=0.0)
            return torch.where(eps < 0, (2 * bound) ** 3.5 * (3 / (7 * math.pi ** 3)), torch.zeros_like(eps))
        eps = kin - M / (R0 + r)
        q2 = torch.clamp(-R0 / M * eps, min=0.0)
        q = torch.sqrt(q2)
        a1 = M / (8 * math.sqrt(2) * (math.pi * R0 * math.sqrt(M / R0)) ** 3) * (1 - q2) ** -2.5
        a2 = 3 * torch.asin(q) + q * torch.sqrt(1 - q2) * (1 - 2 * q2) * (8 * q2 * q2 - 8 * q2 - 3)
        return torch.where(eps < 0, a1 * a2, torch.zeros_like(eps))

    @staticmethod
    def _foot(R, U, J, dt, R0):
        """Straight-line motion a time dt back, as r and v_r, with a mirror at R0 > 0."""
        v2 = U * U + (J / R) ** 2

        def free(R, U, v2, t):  # R(t)^2 = R^2 - 2 R U t + v^2 t^2
            w = R * U - v2 * t
            r = torch.sqrt(w * w + J * J) / torch.sqrt(v2)
            return r, w / r
        r, u = free(R, U, v2, dt)
        if R0 > 0:
            A, B, C = v2, -2 * R * torch.abs(U), R * R - R0 * R0
            D = B * B - 4 * A * C
            root = torch.sqrt(torch.clamp(D, min=0.0))
            t0, t1 = (-B - root) / (2 * A), (-B + root) / (2 * A)
            hit = torch.where(t0 < 0, t1, t0)
            ok = (U > 0) & (D >= 0) & (hit >= 0) & (hit < dt) & (hit < R * torch.abs(U) / v2)
            rh, uh = free(R, U, v2, hit)
            rm, um = free(rh, -torch.abs(uh), uh * uh + (J / rh) ** 2, dt - hit)
            r, u = torch.where(ok, rm, r), torch.where(ok, um, u)
        return r, u

    def _stencil(self, fr, fu, live, points=None):
        """Flat indices and weights of the 4 x 4 coefficients at each foot."""
        x = torch.where(live, torch.log(fr / self.R[0]) * self.hr, torch.zeros_like(fr))
        y = torch.where(live, (fu - self.U[0]) * self.hu, torch.zeros_like(fu))
        nx, ny = x.floor().clamp(0, self.nR - 2), y.floor().clamp(0, self.nU - 2)
        wx, wy = self._weights(x - nx), self._weights(y - ny)
        where = torch.arange(len(fr), device=DEV) if points is None else points
        base = (where // (self.nU * self.nR)) * ((self.nU + 2) * (self.nR + 2))
        base = base + ny.long() * (self.nR + 2) + nx.long()
        return base, wx, [w * live for w in wy]

    @staticmethod
    def _weights(t):
        s = 1 - t
        return [s ** 3 / 6, (1 + 3 * s + 3 * s * s - 3 * s ** 3) / 6,
                (1 + 3 * t + 3 * t * t - 3 * t ** 3) / 6, t ** 3 / 6]

    def _eval(self, c, stencil):
        base, wx, wy = stencil
        out = 0.0
        for a in range(4):
            at = base + a * (self.nR + 2)
            out = out + wy[a] * (wx[0] * c[at] + wx[1] * c[at + 1] + wx[2] * c[at + 2] + wx[3] * c[at + 3])
        return out

    def _moment(self, f):
        cell = 0.25 * (f[:, 1:, 1:] + f[:, 1:, :-1] + f[:, :-1, 1:] + f[:, :-1, :-1])
        m = torch.einsum("jr,j->r", (cell * self.dU[None, :, None]).sum(1), self.weight) * self.dR
        return torch.cat([m, m.new_zeros(1)])

    def mass(self, dM):
        return torch.cat([dM.new_zeros(1), torch.cumsum(dM, 0)[:-1]])

    def _kick(self, f, acc):
        d = torch.matmul(self.invU, f)  # [nJ, nU + 2, nR]
        new = self.U[:, None] + acc[None, :]
        inside = (new > self.U[0]) & (new < self.U[-1])
        y = torch.where(inside, (new - self.U[0]) * self.hu, torch.zeros_like(new))
        n = y.detach().floor().clamp(0, self.nU - 2)
        w = self._weights(y - n)
        n = n.long()
        out = 0.0
        for k in range(4):
            out = out + w[k] * torch.gather(d, 1, (n + k).expand(self.nJ, -1, -1))
        return out * inside

    def _drift(self, f, s, turn):
        c = torch.matmul(self.invU, torch.matmul(f, self.invR.T)).reshape(-1)
        pad = torch.cat([c, c.new_zeros(2 * self.nR + 12)])
        out = self._eval(pad, self.foot)
        if len(self.point):
            slot = self.off + (self.head + self.len - 1) % self.len
            self.vals[s] = self.vals[s].index_copy(0, slot, self._eval(pad, self.back))
            out = out.index_copy(0, self.point, self.vals[s][self.off + self.head])
            if turn:
                self.head = (self.head + 1) % self.len
        return out.reshape(f.shape)

    def step(self):
        last = self.nS - 1
        if not self.linking:
            self.f = [self._drift(f, s, s == last) for s, f in enumerate(self.f)]
        self.dM = self._moment(sum(self.f))
        self.acc = self.mass(self.dM) / self.R ** 2 * self.dt
        self.f = [self._kick(f, self.acc) for f in self.f]
        self.f = [self._drift(f, s, s == last) for s, f in enumerate(self.f)]

    def stats(self):
        dM = self._moment(sum(self.f))
        M = self.mass(dM)
        ep = -float((dM[:-1] * M[:-1] / (0.5 * (self.R[1:] + self.R[:-1]))).sum())
        f = self.f[0]
        v = 0.25 * (f[:, 1:, 1:] + f[:, 1:, :-1] + f[:, :-1, 1:] + f[:, :-1, :-1])
        w = self.weight[:, None, None] * self.dU[None, :, None] * self.dR[None, None, :]
        uc, rc = self.U[:-1] + 0.5 * self.dU, self.R[:-1] + 0.5 * self.dR
        ek = float((w * 0.5 * v * (uc[None, :, None] ** 2 + (self.J[:, None, None] / rc) ** 2)).sum())
        pos = v > 0
        ent = float((w * torch.where(pos, -v * torch.log(torch.where(pos, v, torch.ones_like(v))),
                                     torch.zeros_like(v))).sum())
        return [float(dM.sum()), ek + ep, ek, ep, ent, float((w * v.abs()).sum()), float((w * v * v).sum())]

    def host_f(self):
        f = [x.detach().cpu().numpy() for x in self.f]
        return np.stack(f, -1) if self.nS > 1 else f[0]


def exact(case, seed):
    models = [_Model(cfg) for cfg in _configs(case, seed)]
    kind = case["kind"]
    if kind == "profile":
        m = models[0]
        dM = m._moment(m.f[0])
        vol = 4 * math.pi / 3 * (m.R[1:] ** 3 - m.R[:-1] ** 3)
        rho = torch.cat([dM[:-1] / vol, dM.new_zeros(1)])
        shell = torch.cat([dM[:-1] / (0.5 * (m.R[1:] + m.R[:-1])), dM.new_zeros(1)])
        phi = -(m.mass(dM) / m.R + torch.flip(torch.cumsum(torch.flip(shell, [0]), 0), [0]))
        return {"rho": rho, "phi": phi, "mass": m.mass(dM)}
    if kind in ("run", "ensemble"):
        lines = []
        for n in range(1, case["steps"] + 1):
            for m in models:
                m.step()
            if n % STATS_EVERY == 0 or n == case["steps"]:
                lines.append([m.stats() for m in models])
        if kind == "ensemble":
            return {"f": [m.host_f() for m in models], "stats": np.array(lines)}
        m = models[0]
        return {"f": m.host_f(), "stats": np.array([x[0] for x in lines]), "dM": m.dM, "acc": m.acc,
                "total": float(m.dM.sum())}
    mass, gf, gv = [], [], []
    for m in models:
        if m.nJ * m.nU * m.nR * case["steps"] > 4e8:
            return None  # the graph of torch.autograd would not fit
        target = m.mass(m._moment(m.f[0]))
        f0, v0 = m.f[0].requires_grad_(), m.vals[0].requires_grad_()
        m.f, m.vals = [f0], [v0]
        for _ in range(case["steps"]):
            m.step()
        M = m.mass(m._moment(m.f[0]))
        loss = ((M - target.detach()) ** 2).sum()
        g = torch.autograd.grad(loss, [f0, v0], allow_unused=True)
        mass.append(M.detach())
        gf.append(g[0])
        gv.append(g[1] if g[1] is not None else torch.zeros_like(v0))
    return {"mass": mass, "grad_f0": gf, "grad_vals0": gv}
