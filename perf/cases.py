"""The calls whose speed matters to a user of this library, as named cases with
inputs made from a seed, and the same quantities in plain 64-bit torch.

Every case goes through the Python entry points (magritte_amd.solver and
magritte_amd.autograd) on models of the shapes that the package's generators,
tests and benchmark use: 1D lines, spherically symmetric shells and 3D
jittered-grid winds (Delaunay neighbours, HEALPix rays) of linear rotors or of
blended lines, smooth or clumpy.  The kinds:

* solve: the Feautrier formal solve (u, J and the Lambda diagonal, or J and the
  diagonal alone as the level-population loop needs them);
* gradJ: J and its gradient with respect to the line emissivity and opacity;
* image, imagegrad: the projection-surface image, and an image loss's gradient
  with respect to the log-density and temperature of every point;
* shortchar: the order-0 short-characteristics solve;
* stateq: one statistical-equilibrium update of all level populations;
* batch: many small models in one persistent launch;
* loop: the level-population loop, formal solves and updates alternating.
"""
import math

import numpy as np
import torch

from magritte_amd import _abi, autograd, models, solver

DEV = "cuda:0"


# ---------------------------------------------------------------------------
# the cases


def _solve(name, model, size, nrays, nquads, nlev, precision, u, clumps=0.0, blended=False):
    return dict(name=name, kind="solve", model=model, size=size, nrays=nrays, nquads=nquads,
                nlev=nlev, precision=precision, u=u, clumps=clumps, blended=blended)


def _wind(kind, size, nrays, nquads, nlev, precision, clumps=0.0, **more):
    return dict(kind=kind, model="wind", size=size, nrays=nrays, nquads=nquads, nlev=nlev,
                precision=precision, clumps=clumps, blended=False, **more)


def listed():
    return [
        # the smallest call, as in a first script or a unit test: one line, one ray pair,
        # some hundred points; launches and latency are what it costs
        _solve("line_1d", "line", 101, 2, 31, 2, "fp64", True),
        # a spherically symmetric benchmark model: few points, many rays, the odd
        # quadrature order the 1D non-LTE benchmarks use
        _solve("shells_1d", "shells", 250, 200, 11, 2, "fp64", True),
        # the benchmark's formal solve: 32^3 wind, ten-level rotor, every output kept
        _solve("wind_32_mixed", "wind", 32, 12, 31, 10, "mixed", True),
        # hyperfine-like overlapping lines: several lines in each window, ragged sizes
        _solve("blended_19_fp64", "wind", 19, 48, 23, 6, "fp64", False, blended=True),
        # the formal solve inside a non-LTE loop: many lines, clumps (interpolated
        # segments), J and Lambda only
        _solve("rotor41_18_fp64", "wind", 18, 48, 31, 41, "fp64", False, clumps=0.5),
        # gradient-based inversion from the radiation field: forward and backward
        dict(_wind("gradJ", 24, 12, 31, 10, "fp64"), name="gradient_J_24_fp64"),
        # synthetic observation: one image of the benchmark's wind
        dict(_wind("image", 32, 12, 31, 10, "mixed", pixels=256, nfreqs=31), name="image_256_mixed"),
        # fitting an observation: loss on an image, gradient in (log n, T), clumpy
        dict(_wind("imagegrad", 24, 12, 31, 10, "fp64", clumps=0.5, pixels=128, nfreqs=31),
             name="image_gradient_128_fp64"),
        # the sibling formal solver of the short-characteristics loop
        dict(_wind("shortchar", 20, 12, 31, 10, "fp64", u=True), name="shortchar_20_fp64"),
        # the other half of a non-LTE iteration: 41 levels at every point
        dict(_wind("stateq", 18, 12, 31, 41, "fp64", clumps=0.5), name="stateq41_18"),
        # a survey of small models in one launch
        dict(_wind("batch", 14, 12, 31, 10, "mixed", count=12), name="batch_12_mixed"),
        # a whole small non-LTE run: launches and the loop's own work between the solves
        dict(_wind("loop", 10, 12, 17, 6, "fp64", iterations=3, ng=False), name="nlte_loop_10_fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    cap = max(work(c)["flops"] for c in listed())
    for _ in range(200):
        kind = rng.choice(["solve", "solve", "solve", "solve", "gradJ", "image", "imagegrad",
                           "shortchar", "stateq", "batch", "loop"])
        prec = rng.choice(["fp64", "mixed"])
        if kind == "solve":
            model = rng.choice(["line", "shells", "wind", "wind"])
            if model == "line":
                c = _solve("", model, _log_int(rng, 20, 900), 2, rng.randint(1, 64), 2, prec,
                           rng.random() < 0.5)
            elif model == "shells":
                c = _solve("", model, _log_int(rng, 20, 260), 2 * rng.randint(10, 100),
                           rng.randint(5, 100), 2, prec, rng.random() < 0.5)
            else:
                blended = rng.random() < 0.3
                c = _solve("", model, rng.randint(8, 32), rng.choice([12, 48]), rng.randint(7, 40),
                           rng.randint(2, 8) if blended else rng.randint(2, 41), prec,
                           rng.random() < 0.5, 0.0 if blended else rng.choice([0.0, 0.5]), blended)
        else:
            top = dict(gradJ=24, image=32, imagegrad=24, shortchar=20, stateq=18, batch=14, loop=12)
            c = _wind(kind, rng.randint(6, top[kind]), 12, rng.randint(7, 33),
                      rng.randint(2, 41) if kind == "stateq" else rng.randint(2, 14), prec,
                      rng.choice([0.0, 0.5]))
            if kind in ("image", "imagegrad"):
                c.update(pixels=_log_int(rng, 16, 256 if kind == "image" else 128),
                         nfreqs=rng.randint(3, 64))
            if kind == "shortchar":
                c.update(u=rng.random() < 0.5)
            if kind == "batch":
                c.update(count=rng.randint(3, 16))
            if kind in ("stateq", "loop"):
                c.update(precision="fp64")
            if kind == "loop":
                c.update(iterations=rng.randint(2, 4), ng=rng.random() < 0.5, clumps=0.0)
        c.pop("name", None)
        if work(c)["flops"] <= cap:
            return c
    raise RuntimeError("no case drawn")


def _sizes(case):
    """(points, ray directions, lines, frequencies, mean steps of a half ray)"""
    n, L = case["size"], max(1, case["nlev"] - 1)
    if case["model"] == "line":
        P, steps = n, n / 2
    elif case["model"] == "shells":
        P, steps = n, 0.9 * n
    else:
        P, steps = n**3, 0.41 * n
    return P, case["nrays"], L, L * case["nquads"], steps


def work(case):
    """Each input read and each output written once; about 60 floating-point operations
    per traced segment and frequency of the ray solves (the optical depth, the source
    and one row of the elimination), and the elimination's of the rate matrices."""
    P, R, L, F, steps = _sizes(case)
    mesh = P * (64 + 15 * 4 + 8 * 4)           # positions, velocities, neighbours, per-point data
    inputs = mesh + P * L * 32 + P * F * 8     # line data, frequencies
    ray = P * R * steps * F * 60.0
    kind = case["kind"]
    if kind == "solve":
        return {"bytes": inputs + 8 * P * (F + L) + (8 * P * F * R / 2 if case["u"] else 0), "flops": ray}
    if kind == "shortchar":
        return {"bytes": inputs + 8 * P * (F + L) + (8 * P * F * 2 * R if case["u"] else 0), "flops": ray}
    if kind == "gradJ":  # the backward sweeps do about as much again as the forward, twice
        return {"bytes": 2 * inputs + 8 * P * F * 2 + 16 * P * L, "flops": 3 * ray}
    if kind in ("image", "imagegrad"):
        N, f = case["pixels"] ** 2, case["nfreqs"]
        pix = N * 1.1 * case["size"] * f * 60.0
        out = 8 * N * (f + 2)
        fr = mesh + P * L * 32 + 8 * P
        if kind == "image":
            return {"bytes": fr + out, "flops": pix}
        return {"bytes": 2 * fr + 2 * out + 32 * P * L, "flops": 3 * pix}
    if kind == "stateq":
        return {"bytes": 8 * P * F + 8 * P * (4 * L + 3 * case["nlev"]), "flops": P * (2 / 3 * case["nlev"] ** 3 + 8 * case["nlev"] ** 2)}
    if kind == "batch":
        k = sum((e / case["size"]) ** 3 for e in _edges(case))
        k4 = sum((e / case["size"]) ** 4 for e in _edges(case))
        return {"bytes": k * (inputs + 8 * P * F), "flops": k4 * ray}
    sq = 2 / 3 * case["nlev"] ** 3 + 8 * case["nlev"] ** 2
    return {"bytes": case["iterations"] * (inputs + 16 * P * (F + L) + 24 * P * case["nlev"]),
            "flops": case["iterations"] * (ray + P * sq)}


def _edges(case):
    """the grid edges of a batch's models: from 6 up to size, as they come"""
    n = case["count"]
    return [max(5, case["size"] - (5 * i) % 9) for i in range(n)]


# ---------------------------------------------------------------------------
# inputs


def _model(case, seed, edge=None):
    rng = np.random.Generator(np.random.PCG64([seed, 77]))
    if case["model"] == "line":
        # temperatures, densities and velocity gradients of the same order as the package's line
        return models.model_line_1d(npoints=case["size"], nquads=case["nquads"],
                                    vmax=1.0e4 * rng.uniform(0.5, 2.0),
                                    density=1.0e12 * rng.uniform(0.5, 2.0),
                                    temperature=20.0 * rng.uniform(0.7, 1.5))
    if case["model"] == "shells":
        ld = models.linedata_two_level(179.88e9 * rng.uniform(0.8, 1.2), 1.0e-4)
        return models.model_velocity_gradient_1d(ld, npoints=case["size"], nrays=case["nrays"],
                                                 nquads=case["nquads"], dx=1.0e12,
                                                 dv=40.0 * rng.uniform(0.6, 1.6),
                                                 n_species=1.0e4 * rng.uniform(0.5, 2.0),
                                                 temperature=45.0 * rng.uniform(0.7, 1.5), turb=150.0)
    n = case["size"] if edge is None else edge
    # every wind differs from the smooth one by 10% of density and temperature, point by
    # point; clumps are a log-normal random field on top, correlated over a few points
    dens = np.exp(0.1 * rng.standard_normal(n**3))
    if case["clumps"]:
        dens = dens * models.grf_clumps(n, sigma=case["clumps"], corr_length=1.0 / 10.0,
                                        seed=int(rng.integers(1 << 31)))
    temp = np.exp(0.1 * rng.standard_normal(n**3)) * rng.uniform(0.9, 1.1)
    m = models.model_wind(n_edge=n, nrays=case["nrays"], nquads=case["nquads"], nlev=case["nlev"],
                          seed=int(rng.integers(1 << 31)), v_rot=5.0e3 if case["clumps"] else 0.0,
                          clumps=dens, temp_scale=temp)
    if case["blended"]:
        # lines one to three thermal widths apart
        k = case["nlev"] - 2
        ld = models.linedata_blended(115.0e9, list(np.cumsum(rng.uniform(1.0e-6, 3.0e-6, k))),
                                     A=list(1.0e-7 * rng.uniform(0.5, 2.0, k + 1)))
        ld["colpar"] = [models.colpar_constant(ld, 0, 1.0e-16)]
        m.set_lines([ld], case["nquads"])
        m.finalize()
    return m


def _options(case, m):
    return m.options(precision=_abi.PREC_MIXED if case["precision"] == "mixed" else _abi.PREC_FP64)


def _observation(case, seed, m):
    """direction, frequency grid and target image of the image cases"""
    rng = np.random.Generator(np.random.PCG64([seed, 78]))
    rd = rng.standard_normal(3)
    rd[2] += 0.3
    nu0 = m.line[0] * (1 + rng.uniform(-1e-5, 1e-5))
    fr = m.image_frequencies(nu0 * (1 - 1e-4), nu0 * (1 + 1e-4), case["nfreqs"])
    nu = float(m.line[0])
    level = 2 * models.HH * nu**3 / models.CC_SQUARED / math.expm1(models.HH * nu / (models.KB * 30.0))
    target = level * rng.uniform(0.0, 1.0, (case["pixels"] ** 2, case["nfreqs"]))
    return rd, fr, target


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        ms = [_model(case, seed + 1000 * (i + 1), e) for i, e in enumerate(_edges(case))]
        plan = solver.BatchPlan([solver.DeviceModel(m) for m in ms], _options(case, ms[0]))
        return {"case": case, "plan": plan}
    m = _model(case, seed)
    dm = solver.DeviceModel(m)
    s = {"case": case, "m": m, "dm": dm, "opts": _options(case, m)}
    if kind == "gradJ":
        g = torch.Generator().manual_seed(seed)
        s["J_bar"] = torch.randn((m.npoints, m.nfreqs), dtype=torch.float64, generator=g).to(DEV)
        s["eps"] = dm.tensors["emissivity"].clone().requires_grad_(True)
        s["kap"] = dm.tensors["opacity"].clone().requires_grad_(True)
    if kind in ("image", "imagegrad"):
        s["rd"], s["fr"], target = _observation(case, seed, m)
    if kind == "imagegrad":
        s["target"] = torch.from_numpy(target).to(DEV)
        s["thermo"] = autograd.LineThermo(m, torch.device(DEV))
        s["log_n"] = s["thermo"].log_density().clone().requires_grad_(True)
        s["T"] = s["thermo"].temperature().clone().requires_grad_(True)
    if kind in ("stateq", "loop"):
        s["lp"] = solver.LevelPopulations(dm)
    if kind == "stateq":
        s["pop"] = m.population
        s["J"], s["lam"] = (torch.from_numpy(a).to(DEV) for a in _radiation(case, seed, m))
    return s


def _radiation(case, seed, m):
    """A radiation field and Lambda diagonal of the kind a formal solve hands to the update:
    J between the background's and the local Planck function, by line and point, and
    elements that cancel part of it."""
    rng = np.random.Generator(np.random.PCG64([seed, 79]))
    P, L, Q = m.npoints, m.nlines, m.nquads
    nu = m.nu.reshape(P, L, Q)
    b = lambda T: 2 * models.HH * nu**3 / models.CC_SQUARED / np.expm1(models.HH * nu / (models.KB * T))
    w = rng.uniform(0.05, 0.9, (P, L, 1))
    J = w * b(m.temperature[:, None, None]) + (1 - w) * b(models.T_CMB)
    up = m.population.reshape(P, -1)[:, m.linedata[0]["irad"]]
    Jl = (J * m.quad_weights[0]).sum(axis=2)
    lam = rng.uniform(0.0, 0.5, (P, L)) * Jl / (models.HH / (4 * math.pi) * np.maximum(up, 1e-30))
    return np.ascontiguousarray(J.reshape(P, L * Q)), np.ascontiguousarray(lam)


# ---------------------------------------------------------------------------
# one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "batch":
        return {"J": s["plan"].run()}
    dm, opts = s["dm"], s["opts"]
    if kind == "solve":
        return solver.feautrier_forward(dm, opts, with_u=case["u"])
    if kind == "shortchar":
        return solver.shortchar_forward(dm, opts, with_I=case["u"], with_uv=case["u"])
    if kind == "gradJ":
        s["eps"].grad = s["kap"].grad = None
        J = autograd.formal_solve_J(s["eps"], s["kap"], dm, opts)
        J.backward(s["J_bar"])
        return {"J": J.detach(), "d_eps": s["eps"].grad, "d_kap": s["kap"].grad}
    if kind == "image":
        I, X, Y = solver.image_new(dm, opts, s["rd"], case["pixels"], case["pixels"], s["fr"])
        return {"I": I, "X": X, "Y": Y}
    if kind == "imagegrad":
        s["log_n"].grad = s["T"].grad = None
        I = autograd.image_log_density_temperature(s["log_n"], s["T"], s["thermo"], dm, opts, s["rd"],
                                                   case["pixels"], case["pixels"], s["fr"])
        ((I - s["target"]) ** 2).sum().backward()
        return {"I": I.detach(), "d_log_n": s["log_n"].grad, "d_T": s["T"].grad}
    lp = s["lp"]
    if kind == "stateq":
        lp.set_populations(s["pop"])
        conv, Jl, Je = lp.stateq(s["J"], s["lam"], want_J=True)
    else:
        lp.set_lte()
        solver.compute_level_populations_sparse(dm, opts, lp, use_ng=case["ng"],
                                                max_iterations=case["iterations"])
    pop, _ = lp.populations()
    out = {"pop": pop, "eps": dm.tensors["emissivity"], "kap": dm.tensors["opacity"]}
    if kind == "stateq":
        out.update(J_lin=Jl, J_eff=Je)
    return out


def tolerance(case):
    # About four times and more what the path was seen to be off exact(), whose error functions,
    # exponentials and logarithms are double where the method rounds them to float: that is what
    # another order of the same operations can move.  Errors seen: 2e-8 to 2e-7 of the solves,
    # images and gradients (mixed precision no more than FP64), 1e-6 of the short characteristics'
    # Lambda elements, 1e-13 of the populations after one update and 1e-9 after a few iterations,
    # which an extrapolation (ng) amplifies.
    if case["kind"] == "loop":
        return {"rel": 1e-6, "max": 4e-5} if case["ng"] else {"rel": 1e-8, "max": 4e-7}
    return {"rel": {"shortchar": 5e-6, "stateq": 1e-12}.get(case["kind"], 1e-6)}


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch


class _Ref:
    """The arrays of a model as float64 tensors, and the line data (P, L) in use."""

    def __init__(self, m):
        t = lambda a, dt=torch.float64: torch.as_tensor(np.asarray(a).astype(np.int64) if dt == torch.long else np.asarray(a), dtype=dt, device=DEV)
        self.m = m
        self.P, self.L, self.Q = m.npoints, m.nlines, m.nquads
        self.pos, self.vel = t(m.position), t(m.velocity)
        K = int(m.n_neighbors.max())
        k = np.arange(K)[None, :]
        at = np.minimum(m.cum_n_neighbors[:, None].astype(np.int64) + k, len(m.neighbors) - 1)
        self.nbr = t(m.neighbors[at], torch.long)
        self.has = t(k < m.n_neighbors[:, None], torch.bool)
        self.inner = t(m.point2boundary == m.npoints, torch.bool)
        self.dirs, self.w = t(m.ray_direction.reshape(-1, 3)), t(m.ray_weight)
        self.dsm = t(m.dshift_max)
        u = 2 * models.KB / (models.AMU * models.CC_SQUARED)
        self.ub = torch.sqrt(u * m.max_inverse_mass * t(m.temperature) + t(m.vturb2))
        self.line, self.nu = t(m.line), t(m.nu).reshape(self.P, self.L, self.Q)
        self.set_lines(t(m.emissivity), t(m.opacity), t(m.inverse_width), t(m.interp_crit))
        gap = np.diff(np.sort(m.line)) / m.line.mean() if m.nlines > 1 else np.array([1.0])
        self.blended = bool(gap.min() < 1e-2)
        p = m.params
        self.min_op, self.far = p["min_opacity"], p["max_distance_opacity_contribution"]
        self.log_max = float(np.float32(np.log(np.float32(p["max_interpolation_diff"]))))

    def set_lines(self, eps, kap, iw, crit):
        self.eps, self.kap, self.iw, self.crit = eps, kap, iw, crit

    def planck(self, nu):
        return (2 * models.HH / models.CC_SQUARED) * nu**3 / torch.expm1(models.HH * nu / (models.KB * models.T_CMB))

    def _next(self, o, d, c, Z):
        """the next point on each ray (origin o, direction d) from c at Z; -1: none"""
        if self.m.spherical_symmetry:
            rc, r2 = o @ d, (o * o).sum(1)
            rs2 = r2 - rc * rc
            n2 = lambda p: (self.pos[p] ** 2).sum(1)
            inward = Z < -rc
            lo = (c - 1).clamp(min=0)
            crossing = n2(lo) >= rs2
            hi = (c + 1).clamp(max=self.P - 1)
            dz_in = torch.where(crossing, -torch.sqrt((n2(lo) - rs2).clamp(min=0)) - (rc + Z), -2 * (rc + Z))
            dz_out = torch.sqrt((n2(hi) - rs2).clamp(min=0)) - (rc + Z)
            nxt = torch.where(inward, torch.where(c <= 0, torch.full_like(c, -1), torch.where(crossing, lo, c)),
                              torch.where(c >= self.P - 1, torch.full_like(c, -1), hi))
            return nxt, torch.where(inward, dz_in, dz_out)
        cand = self.nbr[c]
        R = self.pos[cand] - o[:, None, :]
        Zn = R[..., 0] * d[0] + R[..., 1] * d[1] + R[..., 2] * d[2]
        d2 = R[..., 0] ** 2 + R[..., 1] ** 2 + R[..., 2] ** 2 - Zn * Zn
        d2 = torch.where(self.has[c] & (Zn > Z[:, None]), d2, torch.inf)
        best, at = d2.min(dim=1)
        nxt = cand.gather(1, at[:, None])[:, 0]
        return torch.where(torch.isinf(best), -1, nxt), Zn.gather(1, at[:, None])[:, 0] - Z

    def _shift(self, o, vo, d, c, Z):
        """the frequency shift at c of each ray; vo: the velocity it is relative to, or None"""
        if self.m.spherical_symmetry:
            s = self.vel[c, 0] * ((o @ d) + Z) / self.pos[c, 0]
            s = 1 + (s - (vo @ d))
            return torch.where((o * o).sum(1) == 0, torch.ones_like(s), s)
        v = self.vel[c] if vo is None else self.vel[c] - vo
        return 1 + (v[:, 0] * d[0] + v[:, 1] * d[1] + v[:, 2] * d[2])

    def walk(self, start, o, vo, d, Z=None, image=False):
        """steps of the rays: lists of (points, lengths, shifts), each (N), and their count"""
        N = len(start)
        Z = torch.zeros(N, dtype=torch.float64, device=DEV) if Z is None else Z
        c, on = start.clone(), torch.ones(N, dtype=torch.bool, device=DEV)
        n = torch.zeros(N, dtype=torch.long, device=DEV)
        steps, met = [], torch.zeros_like(on)
        centre = torch.as_tensor(self.m.center, device=DEV)
        while True:
            nxt, dz = self._next(o, d, c, Z)
            on = on & (nxt >= 0)
            if not bool(on.any()):
                break
            nxt, dz = torch.where(on, nxt, start), torch.where(on, dz, 0.0)
            Z = Z + dz
            steps.append((nxt, torch.where(on, dz, 1.0), self._shift(o, vo, d, nxt, Z)))
            n += on
            go = self.inner[nxt]
            met = met | (on & go)
            if image:
                go = go | (((self.pos[nxt] - centre) @ d) < 0)
            c = torch.where(on, nxt, c)
            on = on & go
        return steps, n * met if image else n

    def sweep(self, start, shift0, freq, lines, steps, n, m_all, backward, method="feautrier"):
        """One half ray from its outer end to its origin: the last row's X, XI, Y, the last
        depth and source, and whether there is a segment (N, L, Q); for the short
        characteristics, the intensity and the last depth."""
        N = len(start)
        full = lambda v: torch.full(freq.shape, v, dtype=torch.float64, device=DEV)
        X, XI, Y, dprev, Sprev = full(1.0), full(0.5), full(0.0), full(1.0), full(0.0)
        begun = torch.zeros((N, 1, 1), dtype=torch.bool, device=DEV)
        l3 = lambda a, p: a.index_select(0, p)[:, lines][:, :, None]
        for s in range(len(steps) - 1, -1, -1):
            nxt, dZ, sh = steps[s]
            crt = start if s == 0 else steps[s - 1][0]
            shc = shift0 if s == 0 else steps[s - 1][2]
            crt = torch.where(s < n, crt, start)
            diff = torch.abs(torch.log((self.crit[nxt] / self.crit[crt]).float()).double())
            cnt = torch.ceil(diff / self.log_max).clamp(min=1)
            cnt = cnt.max(dim=1, keepdim=True)[0] if m_all else cnt[:, lines]
            top = int((cnt * (s < n)[:, None]).max())
            q = {k: (l3(a, nxt), l3(a, crt)) for k, a in (("e", self.eps), ("k", self.kap), ("w", self.iw))}
            for i in range(top, 0, -1):
                on = ((s < n)[:, None] & (i <= cnt))[:, :, None]
                to, ti = (1 - i / cnt)[:, :, None], (1 - (i - 1) / cnt)[:, :, None]
                dz = (dZ[:, None] / cnt)[:, :, None]
                s_out = sh[:, None, None] + to * (shc - sh)[:, None, None]
                s_in = sh[:, None, None] + ti * (shc - sh)[:, None, None]
                pin = torch.where((i > 1) & (cnt > 1), nxt[:, None], crt[:, None]) if i > 1 else crt[:, None]
                dsm = torch.minimum(self.dsm[nxt][:, None], self.dsm[pin])[:, :, None]
                ubo, ubi = self.ub[nxt][:, None, None], self.ub[pin][:, :, None]
                fo, fi = freq * s_out, freq * s_in
                erf = torch.abs(s_in - s_out) > dsm
                big, small = torch.maximum(fo, fi), torch.minimum(fo, fi)
                W = self.far * big * torch.maximum(ubo, ubi)
                sums = [0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0]
                for k in range(self.L) if self.blended else [None]:
                    g = {a: v if k is None else tuple(x.index_select(1, torch.tensor([k], device=DEV)) for x in v) for a, v in q.items()}
                    line = self.line[lines][None, :, None] if k is None else self.line[k]
                    mix = lambda a, b, t: torch.where(t == 0, a, torch.where(t == 1, b, a * (b / a) ** t))
                    (e1, e2), (k1, k2), (w1, w2) = g["e"], g["k"], g["w"]
                    wo, wi = w1 + (w2 - w1) * to, w1 + (w2 - w1) * ti
                    ko, ki, eo, ei = mix(k1, k2, to), mix(k1, k2, ti), mix(e1, e2, to), mix(e1, e2, ti)
                    So, Si = mix(e1 / k1, e2 / k2, to), mix(e1 / k1, e2 / k2, ti)
                    # line-integrated depth
                    wm = 0.5 * (wo + wi)
                    a, b = (line - fo) * wm, (line - fi) * wm
                    both = torch.minimum(a, b)
                    neg = torch.maximum(a, b)
                    ed = torch.where(both > 0, torch.erfc(a.abs()) - torch.erfc(b.abs()),
                                     torch.where(neg < 0, torch.erfc(b.abs()) - torch.erfc(a.abs()),
                                                 torch.erf(b) - torch.erf(a)))
                    safe = torch.where(erf, b - a, 1.0)
                    dl = dz * (wm * (0.5 * (ko + ki) * ed * 0.5 / safe) + self.min_op)
                    near = ((small - W <= line) & (line <= big + W)).double()
                    sums[0] = sums[0] + near * dl
                    sums[1] = sums[1] + near * dl * So
                    sums[2] = sums[2] + near * dl * Si
                    # emissivity and opacity at the two ends
                    for j, (f, ub, w, e, kk) in enumerate(((fo, ubo, wo, eo, ko), (fi, ubi, wi, ei, ki))):
                        prof = w / math.sqrt(math.pi) * torch.exp(-(w * (f - line)) ** 2)
                        prof = prof * (torch.abs(f - line) <= self.far * f * ub).double()
                        sums[3 + 2 * j] = sums[3 + 2 * j] + prof * e
                        sums[4 + 2 * j] = sums[4 + 2 * j] + prof * kk
                bound = self.min_op * dz
                d_erf = torch.where((sums[0] > -bound) & (sums[0] < bound), bound + 0 * sums[0], sums[0])
                co, ci = sums[4] + self.min_op, sums[6] + self.min_op
                pick = lambda x, y: torch.where(erf, x, y)
                dt = pick(d_erf, 0.5 * (co + ci) * dz)
                S_out, S_in = pick(sums[1] / d_erf, sums[3] / co), pick(sums[2] / d_erf, sums[5] / ci)
                dt = torch.where(on, dt, 1.0)
                if method == "shortchar":
                    Ib = self.planck(freq * s_out)
                    dt = dt.clamp(min=1e-15)
                    prev = torch.where(begun, Y, Ib)
                    new = torch.exp(-dt) * prev + torch.expm1(-dt) / dt * (S_out - S_in * (1 + dt)) + S_out - S_in
                    Y, dprev = torch.where(on, new, Y), torch.where(on, dt, dprev)
                    begun = begun | on
                    continue
                Ib = self.planck(freq * s_out)
                Sr = torch.where(begun, Sprev, S_out) if backward else S_out
                bm = 1 + 2 / dt
                Xb, Yb = 0.5 * bm * dt * dt, (Sr + 2 * Ib / dt) / (bm + 2 / dt / dt)
                avg = 0.5 * (dprev + dt)
                r = 1 / (avg * dprev)
                Xn = (r * X * XI + 1) * avg * dt
                Yn = (r * Y + Sr) / (1 + Xn) * avg * dt
                Xn, Yn = torch.where(begun, Xn, Xb), torch.where(begun, Yn, Yb)
                X, Y = torch.where(on, Xn, X), torch.where(on, Yn, Y)
                XI = torch.where(on, 1 / (1 + Xn), XI)
                dprev, Sprev = torch.where(on, dt, dprev), torch.where(on, S_in, Sprev)
                begun = begun | on
        return X, XI, Y, dprev, Sprev, begun

    def last_row(self, h, Ib):
        """u of the last row, closed by the boundary intensity there"""
        X, _, Y, d, S, _ = h
        a, bm = 2 / (d * d), 1 + 2 / d
        den = (bm + a) * X + bm
        return (a * Y + S + 2 * Ib / d) * (1 + X) / den, (1 + X) / den

    def pair(self, rr, pts, method="feautrier"):
        """u and the diagonal of the inverse at the points pts for one ray pair; for the
        short characteristics both intensities and last depths"""
        ar = int(self.m.antipod[rr])
        lines = torch.arange(self.L, device=DEV)
        freq, half = self.nu[pts], []
        for r, back in ((rr, False), (ar, True)):
            d = self.dirs[r]
            steps, n = self.walk(pts, self.pos[pts], self.vel[pts], d)
            s0 = self._shift(self.pos[pts], self.vel[pts], d, pts, torch.zeros(len(pts), dtype=torch.float64, device=DEV))
            half.append(self.sweep(pts, s0, freq, lines, steps, n, False, back, method))
        Ib = self.planck(freq)
        f, b = half
        if method == "shortchar":
            return [(torch.where(h[5], h[2], Ib), h[3], h[5]) for h in half]
        dc = b[3]
        avg = 0.5 * (f[3] + dc)
        r = 1 / (avg * f[3])
        iC = torch.where(f[5], avg * dc, 0.5 * dc * dc)
        bm = 1 + 2 / dc
        FF = torch.where(f[5], (r * f[0] * f[1] + 1) * avg * dc, bm * iC)
        Su = torch.where(f[5], (r * f[2] + b[4]) / (1 + FF) * iC, (b[4] + 2 * Ib / dc) / (bm + 2 / dc / dc))
        den = 1 / (FF + b[0] * b[1])
        u, lam = (Su * (1 + FF) + b[2]) * den, iC * den
        ul, laml = self.last_row(f, Ib)
        u, lam = torch.where(b[5], u, ul), torch.where(b[5], lam, laml)
        none = ~(b[5] | f[5])
        return torch.where(none, Ib, u), torch.where(none, 0.0, lam)

    def lam_factor(self, wr):
        """what an element of the approximated Lambda operator carries beside the solve's part"""
        wq = torch.as_tensor(self.m.quad_weights[0], device=DEV)
        A = torch.as_tensor(self.m.line_A, device=DEV)[None, :, None]
        chi = self.min_op
        for k in range(self.L) if self.blended else [None]:
            w, kk = (self.iw, self.kap) if k is None else (self.iw[:, k:k + 1], self.kap[:, k:k + 1])
            d = 0.0 * self.line[None, :] if k is None else (self.line - self.line[k])[None, :]
            near = torch.abs(d) <= self.far * self.line[None, :] * self.ub[:, None]
            chi = chi + near * kk * w / math.sqrt(math.pi) * torch.exp(-(w * d) ** 2)
        x = self.iw[:, :, None] * (self.nu - self.line[None, :, None])
        phi = self.iw[:, :, None] / math.sqrt(math.pi) * torch.exp(-x * x)
        return A * wq * wr * self.nu * phi / chi[:, :, None]

    def solve(self, want_u):
        P, F = self.P, self.L * self.Q
        pts = torch.arange(P, device=DEV)
        J, lam, us = 0.0, 0.0, []
        for rr in range(self.m.hnrays):
            w = 2 * float(self.m.ray_weight[rr])
            u, lc = self.pair(rr, pts)
            J = J + w * u
            lam = lam + (self.lam_factor(w) * lc).sum(dim=2)
            if want_u:
                us.append(u.reshape(P, F))
        return {"u": torch.stack(us) if want_u else None, "J": J.reshape(P, F), "lambda_diag": lam}


def _image64(R, case, rd, fr):
    """intensity of the projection-surface image, in R's line data"""
    m = R.m
    d = torch.as_tensor(rd / np.sqrt((rd**2).sum()), device=DEV)
    rx, ry, rz = (float(x) for x in d)
    den = math.sqrt(rx * rx + ry * ry)
    ex = torch.tensor([ry / den, -rx / den, 0.0], dtype=torch.float64, device=DEV)
    ey = torch.tensor([rx * rz / den, ry * rz / den, -den], dtype=torch.float64, device=DEV)
    b = torch.as_tensor(m.boundary2point.astype(np.int64), device=DEV)
    bx, by = R.pos[b] @ ex, R.pos[b] @ ey
    n = case["pixels"]
    cell = lambda v: float(v.min()) + ((float(v.max()) - float(v.min())) / n) * (torch.arange(n, device=DEV, dtype=torch.float64) + 0.5)
    X, Y = cell(bx), cell(by)
    first = int(m.point2boundary[0])
    cand = torch.cat([torch.tensor([first if first < m.npoints else 0], device=DEV), b[1:]])
    z = R.pos[cand] @ d
    begin = cand[int(torch.argmin(z))]
    o = X.repeat_interleave(n)[:, None] * ex + Y.repeat(n)[:, None] * ey + d * float(R.pos[begin] @ d)
    ip = begin.expand(len(o)).clone()
    bdy = ~R.inner
    while True:  # to the boundary point nearest to the pixel's ray, neighbour by neighbour
        def dist(p):
            r = R.pos[p] - o.reshape([len(o)] + [1] * (p.dim() - 1) + [3])
            zr = r @ d
            return (r * r).sum(-1) - zr * zr
        cand = R.nbr[ip]
        far = torch.where(R.has[ip] & bdy[cand], dist(cand), torch.inf)
        best, at = far.min(dim=1)
        better = best < dist(ip)
        if not bool(better.any()):
            break
        ip = torch.where(better, cand.gather(1, at[:, None])[:, 0], ip)
    Z = (R.pos[ip] - o) @ d
    steps, S = R.walk(ip, o, None, d, Z, image=True)
    s0 = R._shift(o, None, d, ip, Z)
    nu = torch.as_tensor(fr["nu"][0], device=DEV)
    freq = nu.expand(len(o), 1, len(nu))
    h = R.sweep(ip, s0, freq, torch.zeros(1, dtype=torch.long, device=DEV), steps, S, True, False)
    Ib = R.planck(freq)
    u, _ = R.last_row(h, R.planck(freq * s0[:, None, None]))
    I = torch.where(h[5], 2 * u - Ib, Ib)[:, 0]
    return I, X.repeat_interleave(n), Y.repeat(n)


def _thermo64(m, log_n, T):
    """line data of the LTE populations of a density and temperature"""
    ld = m.linedata[0]
    t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=DEV)
    tot = t(m.abundance[:, ld["num"]]) * torch.exp(log_n) / t(m.abundance[:, 0])
    x = t(ld["weight"]) * torch.exp(-t(ld["energy"]) / (models.KB * T[:, None]))
    pop = x / x.sum(1, keepdim=True) * tot[:, None]
    eps, kap = _line_data64(m, pop)
    u = 2 * models.KB / (models.AMU * models.CC_SQUARED) * ld["inverse_mass"]
    return eps, kap, 1 / (t(ld["frequency"]) * torch.sqrt(u * T[:, None] + t(m.vturb2)[:, None]))


def _line_data64(m, pop):
    ld = m.linedata[0]
    t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=DEV)
    i, j = (torch.as_tensor(ld[k].astype(np.int64), device=DEV) for k in ("irad", "jrad"))
    c = t(ld["frequency"]) * models.HH / (4 * math.pi)
    return ((c * t(ld["A"]) * pop[:, i]).clamp(min=m.params["min_line_emissivity"]),
            (c * (pop[:, j] * t(ld["Ba"]) - pop[:, i] * t(ld["Bs"]))).clamp(min=m.params["min_line_opacity"]))


def _stateq64(m, pop, J, lam):
    """one statistical-equilibrium update: populations, J_lin, J_eff"""
    ld = m.linedata[0]
    t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=DEV)
    P, n, L = m.npoints, ld["nlev"], ld["nrad"]
    i, j = ([int(x) for x in ld[k]] for k in ("irad", "jrad"))
    jl = (J.reshape(P, L, -1) * t(m.quad_weights[0])).sum(2)
    je = jl - models.HH / (4 * math.pi) * lam * pop[:, i]
    kold = _line_data64(m, pop)[1]
    A = torch.zeros((P, n, n), dtype=torch.float64, device=DEV)

    def rate(I, K, up, down):  # transitions I -> K at rate up, K -> I at rate down, per point
        A[:, K, I] += up
        A[:, K, K] -= down
        A[:, I, K] += down
        A[:, I, I] -= up
    for k in range(L):
        rate(i[k], j[k], ld["A"][k] + ld["Bs"][k] * je[:, k], ld["Ba"][k] * je[:, k])
        rate(i[k], j[k], -lam[:, k] * kold[:, k] / ld["frequency"][k], 0.0)
    for c in ld["colpar"]:
        T, ab = m.temperature, t(m.abundance[:, c["num_col_partner"]])
        tmp = c["tmp"]
        hi = np.clip(np.searchsorted(tmp, T), 0, len(tmp) - 1)
        edge = (hi == 0) | (hi == len(tmp) - 1)
        lo = np.where(edge, hi, hi - 1)
        f = np.where(edge, 0.0, (T - tmp[lo]) / np.where(edge, 1.0, tmp[hi] - tmp[lo]))[:, None]
        Cd, Ce = (t(c[q][lo] + (c[q][hi] - c[q][lo]) * f) * ab[:, None] for q in ("Cd", "Ce"))
        for k, (I, K) in enumerate(zip(c["icol"], c["jcol"])):
            rate(int(I), int(K), Cd[:, k], Ce[:, k])
    tot = t(m.population_tot[0])
    A[:, n - 1, :] = 1.0
    y = torch.zeros((P, n), dtype=torch.float64, device=DEV)
    y[:, n - 1] = tot
    A, y = A.cpu(), y.cpu()
    x = torch.linalg.solve(A, y)
    x = x + torch.linalg.solve(A, y - (A @ x[:, :, None])[:, :, 0])
    x = x.to(DEV).clamp(min=0.0)
    return x * (tot / x.sum(1))[:, None], jl, je


def exact(case, seed):
    kind = case["kind"]
    P, R_, L, F, steps = _sizes(case)
    if kind == "batch":
        return {"J": [_Ref(_model(case, seed + 1000 * (i + 1), e)).solve(False)["J"] if case["clumps"] == 0 or e < 12 else None
                      for i, e in enumerate(_edges(case))]}
    m = _model(case, seed)
    # tens of thousands of small torch operations: left out where they take too long
    slow = P * R_ * steps * F * (8.0 if case["clumps"] else 1.0) * (L if case["blended"] else 1) > 6e10
    if slow and kind in ("solve", "gradJ", "shortchar"):
        return None
    R = _Ref(m)
    if kind == "solve":
        return R.solve(case["u"])
    if kind == "shortchar":
        pts = torch.arange(P, device=DEV)
        I, u, v, J, lam = [None] * m.nrays, [], [], 0.0, 0.0
        for rr in range(m.hnrays):
            w = float(m.ray_weight[rr])
            (a, da, ha), (b, db, hb) = R.pair(rr, pts, "shortchar")
            I[rr], I[int(m.antipod[rr])] = a.reshape(P, F), b.reshape(P, F)
            u.append((0.5 * (a + b)).reshape(P, F))
            v.append((0.5 * (a - b)).reshape(P, F))
            J = J + 2 * w * u[-1]
            f = lambda d, h: torch.where(h, 1 + torch.expm1(-d) / d, 0.0)
            lam = lam + (R.lam_factor(w) * (f(da, ha) + f(db, hb))).sum(2)
        keep = case["u"]
        return {"I": torch.stack(I) if keep else None, "u": torch.stack(u) if keep else None,
                "v": torch.stack(v) if keep else None, "J": J, "lambda_diag": lam}
    if kind == "gradJ":
        g = torch.Generator().manual_seed(seed)
        J_bar = torch.randn((P, F), dtype=torch.float64, generator=g).to(DEV).reshape(P, L, -1)
        eps, kap = R.eps.clone().requires_grad_(True), R.kap.clone().requires_grad_(True)
        J = torch.zeros_like(J_bar)
        for c in torch.arange(P, device=DEV).split(max(64, int(1.2e6 / F))):
            for rr in range(m.hnrays):
                R.set_lines(eps, kap, R.iw, R.crit)
                u, _ = R.pair(rr, c)
                Jp = 2 * float(m.ray_weight[rr]) * u
                (Jp * J_bar[c]).sum().backward()
                J[c] += Jp.detach()
        return {"J": J, "d_eps": eps.grad, "d_kap": kap.grad}
    if kind in ("image", "imagegrad"):
        rd, fr, target = _observation(case, seed, m)
        if kind == "image":
            I, X, Y = _image64(R, case, rd, fr)
            return {"I": I, "X": X, "Y": Y}
        if case["pixels"] ** 2 * case["size"] * case["nfreqs"] > 1.4e7:
            return None
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=DEV)
        log_n, T = torch.log(t(m.abundance[:, 0])).requires_grad_(True), t(m.temperature).requires_grad_(True)
        R.set_lines(*_thermo64(m, log_n, T), R.crit)
        I, _, _ = _image64(R, case, rd, fr)
        ((I - t(target)) ** 2).sum().backward()
        return {"I": I.detach(), "d_log_n": log_n.grad, "d_T": T.grad}
    pop = torch.as_tensor(m.population, device=DEV).reshape(P, -1)
    if kind == "stateq":
        J, lam = (torch.as_tensor(a, device=DEV) for a in _radiation(case, seed, m))
        pop, jl, je = _stateq64(m, pop, J, lam)
        eps, kap = _line_data64(m, pop)
        return {"pop": pop, "eps": eps, "kap": kap, "J_lin": jl, "J_eff": je}
    if case["ng"]:
        return None  # extrapolations amplify the last digits of what they extrapolate
    for _ in range(case["iterations"]):
        out = R.solve(False)
        pop, _, _ = _stateq64(m, pop, out["J"], out["lambda_diag"])
        eps, kap = _line_data64(m, pop)
        R.set_lines(eps, kap, R.iw, kap / torch.as_tensor(m.population_tot[0], device=DEV)[:, None])
    return {"pop": pop, "eps": eps, "kap": kap}
