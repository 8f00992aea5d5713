"""The calls whose speed is tracked, over the sizes a user of the library runs.

A case is one pass of a user's program through gliomasolver_amd's public entry
points.  Kinds (the sizes are those of bench.py, tests/ and apps/):

  forward        a uniform tumour solve from a stored initial state: rd_steps,
                 then the field (bench.py's step; apps/brain.cpp without -adaptive)
  two_pass       the operator and the update called step by step, as
                 apps/rd_pipeline.cpp does (rd_rhs, rd_update, the field)
  likelihood     -logL of the current state against fixed observations
  adjoint        forward + likelihood + six gradients of one solve
  generation     one TMCMC generation as apps/tmcmc_glioma.cpp evaluates it:
                 set_samples, run, likelihood of every sample
  gradients      a population's loss and gradients on mixed grids
  adaptive_steps a multi-level grid stepped between two adaptations
  adaptive_run   a run resumed from stored leaves and fields: constants, then
                 epochs of steps, refinement and compression

Inputs are made from the seed alone: an analytic brain (folded cortex, white
matter, ventricles, no tissue outside the head) and a tumour in its white
matter.  exact() restates the model in 64 bits with torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gliomasolver_amd as gh

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
CUBE_CM = 17.6                            # side of the domain (bench.py)
LIK = (0.0025, 1.0, 0.7, 0.25, 2.0)       # PET variance and scale, T1Gd / FLAIR thresholds, slope
REFINE, COMPRESS = 1e-4, 1e-6             # tolerances of the adaptive workload


def listed():
    return [
        # the smallest call: a coarse solve, bound by launches and the field's way back
        {"name": "forward-32-f32", "kind": "forward", "n": 32, "real": "f32", "steps": 87, "tuned": False},
        # 64^3 in double to T = 300 days, as brain runs it: no tuning call
        {"name": "forward-64-f64", "kind": "forward", "n": 64, "real": "f64", "steps": 344, "tuned": False},
        # the headline solve: 128^3 to T = 400 days with the schedule tuned beforehand
        {"name": "forward-128-f32", "kind": "forward", "n": 128, "real": "f32", "steps": 1971, "tuned": True},
        # a fine grid whose states do not fit the caches
        {"name": "forward-256-f32", "kind": "forward", "n": 256, "real": "f32", "steps": 250, "tuned": True},
        # callers that keep the reference's two passes per step
        {"name": "two-pass-128-f32", "kind": "two_pass", "n": 128, "real": "f32", "steps": 25},
        # one likelihood of a state on the device, every voxel, PET on the 3-voxel lattice
        {"name": "likelihood-128-f32", "kind": "likelihood", "n": 128, "real": "f32", "step_pet": 3,
         "radius": 0.11},
        # gradients of a 64^3 double solve and of the headline solve
        {"name": "adjoint-64-f64", "kind": "adjoint", "n": 64, "real": "f64", "steps": 344, "every": 64},
        {"name": "adjoint-128-f32", "kind": "adjoint", "n": 128, "real": "f32", "steps": 1001, "every": 64},
        # a TMCMC generation on a grid that is no power of two, data of another size
        {"name": "generation-96-f32", "kind": "generation", "bpd": 12, "real": "f32", "samples": 24, "days": 120.0},
        # a population's gradients on 64^3 / 96^3 / 128^3 grids
        {"name": "gradients-mixed-f32", "kind": "gradients", "bpd": 8, "real": "f32", "samples": 12, "days": 250.0,
         "every": 32},
        # levels 3-5, a grown tumour, the steps of five epochs
        {"name": "adaptive-steps-f32", "kind": "adaptive_steps", "top": 5, "real": "f32", "radius": 0.17, "steps": 50},
        # levels 3-5, a small tumour, four epochs of ten steps with refinement and compression
        {"name": "adaptive-run-f32", "kind": "adaptive_run", "top": 5, "real": "f32", "radius": 0.09, "epochs": 4},
    ]


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["forward", "forward", "two_pass", "likelihood", "adjoint", "generation", "gradients",
                       "adaptive_steps", "adaptive_run"])
    real = rng.choice(["f32", "f32", "f64"])
    n = rng.choice([16, 32, 64, 128])
    some = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    span = lambda size, days: max(3, math.ceil(days * size * size / 3750))  # noqa: E731  steps of so many days
    if kind == "forward":
        return {"kind": kind, "n": n, "real": real, "steps": min(1200, span(n, rng.uniform(20, 400))),
                "tuned": rng.random() < 0.5}
    if kind == "two_pass":
        return {"kind": kind, "n": n, "real": real, "steps": some(3, 60)}
    if kind == "likelihood":
        return {"kind": kind, "n": n, "real": real, "step_pet": rng.choice([1, 2, 3]),
                "radius": round(rng.uniform(0.06, 0.14), 3)}
    if kind == "adjoint":
        n = min(n, 64)
        return {"kind": kind, "n": n, "real": real, "steps": span(n, rng.uniform(40, 300)),
                "every": rng.choice([16, 32, 64])}
    if kind == "generation":
        return {"kind": kind, "bpd": rng.randint(3, 11), "real": real, "samples": some(3, 40),
                "days": round(rng.uniform(20.0, 100.0), 1)}
    if kind == "gradients":
        return {"kind": kind, "bpd": rng.randint(3, 7), "real": real, "samples": some(3, 16),
                "days": round(rng.uniform(50.0, 200.0), 1), "every": rng.choice([16, 32, 64])}
    if kind == "adaptive_steps":
        return {"kind": kind, "top": rng.choice([4, 5]), "real": real, "radius": round(rng.uniform(0.06, 0.2), 3),
                "steps": some(5, 60)}
    return {"kind": kind, "top": rng.choice([4, 5]), "real": real, "radius": round(rng.uniform(0.06, 0.14), 3),
            "epochs": rng.randint(1, 5)}


# ---- inputs ------------------------------------------------------------------

class Brain:
    """An analytic head in the unit cube; tissues() at any coordinates."""

    def __init__(self, seed, cells, octant=False):
        r = np.random.default_rng(seed)
        self.c = 0.5 + r.uniform(-0.015, 0.015, 3)
        self.k = r.uniform(2.0, 5.0, (6, 3)) * r.choice([-1.0, 1.0], (6, 3))
        self.ph = r.uniform(0, 2 * np.pi, 6)
        self.sharp = 0.22 * cells  # partial volumes over about two cells
        while True:  # a tumour centre in white matter
            d = r.normal(size=3)
            if octant:  # in the middle of one of the head's octants: the same tiling whatever the seed
                self.tumour = 0.5 + 0.125 * np.where(d < 0, -1.0, 1.0)
            else:
                self.tumour = self.c + 0.5 * np.array([0.40, 0.34, 0.36]) * d / np.linalg.norm(d) * r.uniform(0.6, 1.0)
            p = torch.from_numpy(self.tumour)
            if float(self.tissues(p[0], p[1], p[2])[1]) > 0.95:
                break

    def tissues(self, x, y, z):
        """(gm, wm, csf) fractions."""
        cx, cy, cz = self.c
        ball = lambda o, a: (((x - o[0]) / a[0]) ** 2 + ((y - o[1]) / a[1]) ** 2 + ((z - o[2]) / a[2]) ** 2).sqrt()  # noqa: E731
        e = ball((cx, cy, cz), (0.40, 0.34, 0.36))
        fold = sum(0.02 * torch.sin(2 * math.pi * (k[0] * x + k[1] * y + k[2] * z) + p) for k, p in zip(self.k, self.ph))
        ramp = lambda v: (v * self.sharp + 0.5).clamp(0, 1)  # noqa: E731
        head, cortex, white = ramp(0.36 * (1 - e)), ramp(0.36 * (0.93 + 0.4 * fold - e)), ramp(0.36 * (0.76 + fold - e))
        vent = torch.maximum(ramp(0.06 * (1 - ball((cx - 0.06, cy, cz), (0.03, 0.11, 0.06)))),
                             ramp(0.06 * (1 - ball((cx + 0.06, cy, cz), (0.03, 0.11, 0.06)))))
        cortex = torch.maximum(cortex, white)
        wm, gm = white * (1 - vent), (cortex - white) * (1 - vent)
        return gm, wm, (head - gm - wm).clamp(0, 1)

    def grown(self, x, y, z, radius):
        """A grown tumour's density: a front of the given radius in tissue."""
        gm, wm, csf = self.tissues(x, y, z)
        r = ((x - self.tumour[0]) ** 2 + (y - self.tumour[1]) ** 2 + (z - self.tumour[2]) ** 2).sqrt()
        u = 0.97 * torch.sigmoid((radius - r) / 0.011) * (gm + wm) * (csf <= gm + wm)
        return torch.where(u < 1e-12, torch.zeros_like(u), u)


def lattice(nx, ny=None, nz=None):
    """x, y, z in [0, 1) of an (nz, ny, nx) array, 1 / max(n) apart."""
    ny, nz = ny or nx, nz or nx
    a = [torch.arange(m, device=DEV, dtype=F64) / max(nx, ny, nz) for m in (nz, ny, nx)]
    z, y, x = torch.meshgrid(*a, indexing="ij")
    return x, y, z


def voted(gm, wm, csf):
    """p_w, p_g of the reference's initial condition."""
    t = gm + wm
    keep = ((csf <= t) | (t >= 1)) & (t > 0)
    t = torch.where(keep, t, torch.ones_like(t))
    return torch.where(keep, wm / t, 0.0), torch.where(keep, gm / t, 0.0)


def gaussian(n, centre, pw, pg):
    """The seed tumour: sigma one cell, peak 0.1, in tissue."""
    x, y, z = (n * v for v in lattice(n))
    d2 = (x - centre[0]) ** 2 + (y - centre[1]) ** 2 + (z - centre[2]) ** 2
    return torch.where(pw + pg > 0, 0.1 * torch.exp(-d2 / 2), 0.0)


def observations(brain, n, seed, radius=0.1):
    """T1Gd and FLAIR masks with 5 % of the voxels flipped, PET inside T1Gd."""
    r = np.random.default_rng([seed, 7])
    u = brain.grown(*lattice(n), radius).cpu().numpy()
    t1, fl = (u >= 0.7).astype(np.float64), (u >= 0.25).astype(np.float64)
    for m in (t1, fl):
        f = r.random(m.shape) < 0.05
        m[f] = 1 - m[f]
    return t1, fl, np.where(t1 > 0, u + r.normal(0, 0.05, u.shape), 0.0)


def np_type(case):
    return np.float32 if case["real"] == "f32" else np.float64


def scales(seed, n, case):
    """Dw / L^2, rho and the stable time step of a uniform solve."""
    r = np.random.default_rng([seed, 3])
    Dw = math.exp(r.uniform(math.log(0.008), math.log(0.015))) / CUBE_CM ** 2
    rho = math.exp(r.uniform(math.log(0.02), math.log(0.06)))
    return float(np_type(case)(Dw)), float(np_type(case)(rho)), float(np_type(case)(0.9 / (6 * n * n * Dw)))


def uniform(case, seed):
    """The host arrays of a uniform case."""
    n = case["n"]
    b = Brain(seed, n)
    gm, wm, csf = b.tissues(*lattice(n))
    pw, pg = voted(gm, wm, csf)
    centre = [float(v) for v in np.round(b.tumour * n)]
    if case["kind"] == "likelihood":
        phi = b.grown(*lattice(n), case["radius"])
    else:
        phi = gaussian(n, centre, pw, pg)
    phi = phi.cpu().numpy().astype(np_type(case))
    return b, [a.cpu().numpy() for a in (gm, wm, csf)], phi, centre


def population(case, seed):
    """Anatomies and sample rows of a batched case."""
    r = np.random.default_rng([seed, 5])
    bpds = [case["bpd"]] if case["kind"] == "generation" else [case["bpd"], (3 * case["bpd"]) // 2, 2 * case["bpd"]]
    anat = []
    for i, bpd in enumerate(bpds):
        n = 8 * bpd
        if case["kind"] == "generation":  # scans of another size than the grid
            shape = (n + n // 7, n - n // 9, n + 3)  # nx, ny, nz
        else:
            shape = (n, n, n)
        b = Brain(seed + 101 * i, max(shape))
        data = [a.cpu().numpy() for a in b.tissues(*lattice(*shape))]
        anat.append((bpd, b, data, observations(b, n, seed + 101 * i)))
    m = case["samples"]
    which = r.integers(0, len(bpds), m).astype(np.int32)
    Dw = np.exp(r.uniform(math.log(0.002), math.log(0.015), m))
    rho = np.exp(r.uniform(math.log(0.02), math.log(0.1), m))
    T = case["days"] * r.uniform(0.4, 1.0, m)
    jit = r.uniform(-0.02, 0.02, (m, 3))
    rows, steps = np.zeros((m, 6)), np.zeros(m, np.int64)
    for i in range(m):
        bpd, b = anat[which[i]][:2]
        n = 8 * bpd
        c = b.tumour + jit[i]
        if case["kind"] == "generation":
            rows[i] = (Dw[i], rho[i], T[i], *c)
        else:
            d = Dw[i] / CUBE_CM ** 2
            steps[i] = math.ceil(T[i] * 6 * d * n * n / 0.9)
            rows[i] = (d, rho[i], T[i], *np.round(c * n))
    return anat, which, rows, steps


def leaves_of(case, centre):
    """Rows (level, x, y, z) in canonical order of a 2:1 tiling with levels
    top - 2 .. top, finest where the tumour is."""
    top = case["top"]
    low = top - 2
    reach = case["radius"] + 0.05
    cut = {}
    deeper = None
    for L in range(top - 1, low - 1, -1):  # blocks of level L that are subdivided
        m = 1 << L
        i = np.arange(m)
        d = [np.maximum(0, np.maximum(i / m - centre[a], centre[a] - (i + 1) / m)) ** 2 for a in range(3)]
        c = (d[2][:, None, None] + d[1][None, :, None] + d[0][None, None, :]) < reach ** 2
        if deeper is not None:  # the finer level's subdivided blocks and all their neighbours exist
            w = deeper
            for a in range(3):
                w = w | np.roll(w, 1, a) | np.roll(w, -1, a)
            c = c | w.reshape(m, 2, m, 2, m, 2).any((1, 3, 5))
        cut[L] = deeper = c
    rows = []
    exists = np.ones((1 << low,) * 3, bool)
    for L in range(low, top + 1):
        leaf = exists & ~cut[L] if L < top else exists
        z, y, x = np.nonzero(leaf)
        rows.append(np.stack([np.full_like(x, L), x, y, z], 1))
        if L < top:
            exists = np.repeat(np.repeat(np.repeat(exists & cut[L], 2, 0), 2, 1), 2, 2)
    return np.concatenate(rows).astype(np.int32)


def adapted(case, seed):
    """Leaves and block-major fields phi, p_w, p_g, p_csf of a multi-level case."""
    cells = 8 << case["top"]
    b = Brain(seed, cells, octant=True)
    rows = leaves_of(case, b.tumour)
    t = torch.from_numpy(rows).to(DEV, F64)
    i = torch.arange(8, device=DEV, dtype=F64) / 8
    w = torch.exp2(-t[:, 0])
    at = lambda a, view: ((t[:, a, None] + i) * w[:, None]).reshape(view)  # noqa: E731
    nb = len(rows)
    x, y, z = torch.broadcast_tensors(at(1, (nb, 1, 1, 8)), at(2, (nb, 1, 8, 1)), at(3, (nb, 8, 1, 1)))
    gm, wm, csf = b.tissues(x, y, z)
    pw, pg = voted(gm, wm, csf)
    phi = b.grown(x, y, z, case["radius"])
    fields = [a.cpu().numpy().astype(np_type(case)) for a in (phi, pw, pg, (csf > gm + wm).to(F64))]
    n = cells
    Dw = 0.013 / CUBE_CM ** 2
    return rows, fields, Dw, 0.025, float(np_type(case)(0.9 / (6 * n * n * Dw)))


FIELDS = (gh.FIELD_PHI, gh.FIELD_PW, gh.FIELD_PG, gh.FIELD_PCSF)


def restore(ctx, rows, fields):
    ctx.grid_init_leaves(rows[:, 0], rows[:, 1:])
    for f, v in zip(FIELDS, fields):
        ctx.set_field_blocks(f, v)


# ---- the interface -----------------------------------------------------------

def prepare(case, seed):
    kind, real = case["kind"], case["real"]
    s = {"case": case}
    if kind in ("generation", "gradients"):
        anat, s["which"], s["rows"], s["steps"] = population(case, seed)
        s["batch"] = b = gh.Batch(0, real)
        for bpd, _, data, obs in anat:
            b.set_observations(b.add_anatomy(bpd, *data), *obs)
        return s
    s["ctx"] = ctx = gh.Context(0, real)
    if kind in ("adaptive_steps", "adaptive_run"):
        rows, fields, Dw, rho, s["dt"] = adapted(case, seed)
        ctx.grid_configure(4, case["top"], case["top"] - 2)
        restore(ctx, rows, fields)
        ctx.rd_prepare(Dw, 0.1 * Dw, rho)
        ctx.checkpoint_save(0)
        s.update(rows=rows, fields=fields, D=(Dw, 0.1 * Dw, rho), used=0)
        m = 3 * len(rows)
        s["room"] = (np.zeros(m, np.int32), np.zeros((m, 3), np.int32), np.zeros((m, 8, 8, 8), np_type(case)))
        return s
    n = case["n"]
    brain, anatomy, phi, centre = uniform(case, seed)
    Dw, rho, dt = scales(seed, n, case)
    ctx.grid_init_uniform(n // 8)
    ctx.set_anatomy(*anatomy)
    ctx.set_field(gh.FIELD_PHI, phi)
    ctx.rd_prepare(Dw, 0.1 * Dw, rho)
    if kind in ("likelihood", "adjoint"):
        ctx.lik_set_data(*observations(brain, n, seed))
    if case.get("tuned"):
        ctx.rd_autotune(dt, 20)
    ctx.checkpoint_save(0)
    s.update(dt=dt, centre=centre)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "generation":
        b = s["batch"]
        b.set_samples(s["which"], s["rows"])
        b.run()
        return b.likelihood(LIK, stepPET=3)
    if kind == "gradients":
        b = s["batch"]
        b.set_adjoint_samples(s["which"], s["rows"], s["steps"])
        loss, grad, _ = b.adjoint(LIK, ckpt_every=c["every"])
        return {"loss": loss, **{"grad%d" % q: np.ascontiguousarray(grad[:, q]) for q in range(6)}}
    ctx = s["ctx"]
    if kind == "likelihood":
        nll, parts, npet = ctx.likelihood(LIK, stepPET=c["step_pet"])
        return {"terms": np.array([nll, *parts]), "points": npet}
    if kind == "adaptive_run":
        restore(ctx, s["rows"], s["fields"])
        ctx.rd_prepare(*s["D"])
        for _ in range(c["epochs"]):
            ctx.rd_steps(10, s["dt"])
            ctx.refine(REFINE, 1)
            ctx.compress(COMPRESS, -1)
        nb = ctx.nblocks()  # into the program's arrays, which have room for more blocks than there are
        room = s["room"]
        for a, v in zip(room, (*ctx.blocks(), ctx.get_field_blocks(gh.FIELD_PHI))):
            a[:nb] = v
            a[nb:s["used"]] = 0
        s["used"] = nb
        return [nb, *room]
    ctx.checkpoint_load(0)
    if kind == "adjoint":
        loss, grad = ctx.rd_adjoint(c["steps"], c["steps"] * s["dt"], s["centre"], 1.0, c["every"], LIK)
        return {"loss": loss, **{"grad%d" % q: grad[q:q + 1] for q in range(6)}}
    if kind == "two_pass":
        for _ in range(c["steps"]):
            ctx.rd_rhs()
            ctx.rd_update(s["dt"])
        return ctx.get_field(gh.FIELD_PHI)
    ctx.rd_steps(c["steps"], s["dt"])
    return ctx.get_field_blocks(gh.FIELD_PHI) if kind == "adaptive_steps" else ctx.get_field(gh.FIELD_PHI)


STEP_FLOPS = 45      # operator and update, per cell
REVERSE_FLOPS = 70   # transposed stencil and the two gradient sums, per cell


def work(case):
    """Inputs once, outputs once; the operations of every cell and step."""
    size = 4 if case["real"] == "f32" else 8
    kind = case["kind"]
    if kind in ("generation", "gradients"):
        _, which, rows, steps = _plan(case)
        cells = sum(c for c, _ in which)
        if kind == "generation":
            return {"bytes": cells * (3 * size + 10), "flops": sum(c * n for c, n in which) * STEP_FLOPS}
        return {"bytes": cells * (3 * size + 10), "flops": sum(c * n for c, n in which) * (STEP_FLOPS + REVERSE_FLOPS)}
    if kind.startswith("adaptive"):
        cells = 512 * len(leaves_of(case, (0.375, 0.375, 0.375)))
        steps = case["steps"] if kind == "adaptive_steps" else 10 * case["epochs"]
        return {"bytes": cells * size * (4 if kind == "adaptive_steps" else 5), "flops": cells * steps * STEP_FLOPS}
    cells = case["n"] ** 3
    if kind == "likelihood":
        return {"bytes": cells * (size + 2 + 8 / case["step_pet"] ** 3), "flops": cells * 50}
    per = STEP_FLOPS + (REVERSE_FLOPS if kind == "adjoint" else 0)
    return {"bytes": cells * (4 * size + (10 if kind == "adjoint" else 0)), "flops": cells * case["steps"] * per}


def _plan(case):
    """(cells, steps) of the samples of a batched case, on average over seeds."""
    bpds = [case["bpd"]] if case["kind"] == "generation" else [case["bpd"], (3 * case["bpd"]) // 2, 2 * case["bpd"]]
    out = []
    for i in range(case["samples"]):
        n = 8 * bpds[i % len(bpds)]
        L = 0.1 * (n + n // 7) if case["kind"] == "generation" else CUBE_CM
        cfl = 0.99 if case["kind"] == "generation" else 0.9
        out.append((n ** 3, math.ceil(0.7 * case["days"] * 6 * 0.0065 / L ** 2 * n * n / cfl)))
    return None, out, None, None


# ---- the model in 64 bits ------------------------------------------------------

def harmonic(a, b):
    s = a + b
    return torch.where(s < 1e-8, 0.0, 2 * a * b / torch.where(s < 1e-8, 1.0, s))


class Model:
    """The operator on a periodic n^3 grid, arrays (..., z, y, x)."""

    def __init__(self, pw, pg, Dw, rho, n):
        self.t, self.rho, self.ih2 = pw + pg, rho, float(n * n)
        df = pw * Dw + pg * (0.1 * Dw)
        self.D = []  # -x, +x, -y, +y, -z, +z
        for a in (-1, -2, -3):
            up = harmonic(torch.roll(df, -1, a), df)
            self.D += [torch.roll(up, 1, a), up]

    AXES = ((-1, 1), (-1, -1), (-2, 1), (-2, -1), (-3, 1), (-3, -1))  # axis and roll that fetch neighbour i

    def flags(self, u):
        return ((u + self.t) < 0.1).to(F64) + 1, (u + self.t) > 0  # 2 where outside, in the domain

    def flux(self, u, o):
        """ih2 sum d'(u_n - u) and ih2 sum d'."""
        s = torch.zeros_like(u)
        d = torch.zeros_like(u)
        for i, (a, r) in enumerate(self.AXES):
            dp = self.D[i] * torch.roll(o, -r, a)  # doubled where the opposite neighbour is outside
            s.addcmul_(dp, torch.roll(u, r, a))
            d += dp
        return (s - d * u) * self.ih2, d * self.ih2

    def step(self, u, dt):
        o, dom = self.flags(u)
        f = self.flux(u, o)[0]
        return (u + dt * torch.where(dom, f + self.rho * u * (1 - u), 0.0)).clamp(0, 1)

    def reverse(self, u, lam, dt):
        """lambda_k before its own mask from the masked lambda_{k+1}; the sums A and B."""
        o, dom = self.flags(u)
        f, d = self.flux(u, o)
        w = torch.where(dom, lam, 0.0)
        acc = torch.zeros_like(u)
        for i, (a, r) in enumerate(self.AXES):
            acc += torch.roll(w, r, a) * self.D[i] * torch.roll(o, 2 * r, a)
        A, B = float((w * f).sum()), float((w * u * (1 - u)).sum())
        return torch.where(dom, lam * (1 + dt * (self.rho * (1 - 2 * u) - d)), lam) + dt * self.ih2 * acc, A, B


def log_bernoulli(u, y, uc):
    d = u - uc
    w2 = torch.where(d > 0, 1.0, d * d)
    al = 0.5 + 0.5 * torch.sign(d) * (1 - torch.exp(-w2 / LIK[4]))
    return torch.where(y, torch.log(al), torch.log(1 - al)).sum()


def likelihood64(u, obs, step_pet):
    """[-logL, PET, T1, T2, points] and dJ/du."""
    t1, fl, pet = (torch.from_numpy(a).to(DEV) for a in obs)
    on = torch.zeros_like(pet, dtype=torch.bool)
    on[::step_pet, ::step_pet, ::step_pet] = True
    on &= pet > 0
    npet = int(on.sum())
    res = torch.where(on, u - LIK[1] * pet, 0.0)
    p = -0.5 * npet * math.log(2 * math.pi * LIK[0]) - 0.5 / LIK[0] * float((res ** 2).sum())
    l1, l2 = (float(log_bernoulli(u, y == 1, c)) for y, c in ((t1, LIK[2]), (fl, LIK[3])))
    g = res / LIK[0]
    for y, c in ((t1, LIK[2]), (fl, LIK[3])):
        d = u - c
        a = 0.5 * torch.exp(-d * d / LIK[4])
        da = a * (-2 * d / LIK[4])
        g -= torch.where(d < 0, torch.where(y == 1, da / a, -da / (1 - a)), 0.0)
    return [-(p + l1 + l2), p, l1, l2, npet], g


def adjoint64(m, u, steps, T, obs, centre, Dw):
    """Loss and the six gradients of one solve."""
    dt = T / steps
    tape = [u]
    for _ in range(steps):
        tape.append(m.step(tape[-1], dt))
    loss, lam = likelihood64(tape[-1], obs, 1)
    A = B = 0.0
    for k in range(steps - 1, -1, -1):
        lam, a, b = m.reverse(tape[k], lam * (tape[k + 1] < 1), dt)
        A, B = A + a, B + b
    x, y, z = (u.shape[-1] * v for v in lattice(u.shape[-1]))
    ic = [float((lam * u * (v - c)).sum()) for v, c in zip((x, y, z), centre)]
    return loss[:4], [dt * A / Dw, dt * B, (A + m.rho * B) / steps, *ic]


def on_grid(bpd, data, real):
    """Scans of any size on the cells of a uniform grid: nearest voxel, as the
    initial condition places cells in Real."""
    t = np.float32 if real == "f32" else np.float64
    i = np.arange(8 * bpd)
    dil = t(1.0 / bpd)
    x = ((i // 8).astype(t) * dil + (dil / t(8)) * (i % 8).astype(t)).astype(np.float64)
    vox = np.floor(x / (1.0 / max(data[0].shape))).astype(int)
    out = []
    for a in data:
        v = torch.zeros((8 * bpd,) * 3, device=DEV, dtype=F64)
        ok = [np.nonzero(vox < m)[0] for m in a.shape]
        v[np.ix_(*ok)] = torch.from_numpy(a[np.ix_(*(vox[k] for k in ok))]).to(DEV)
        out.append(v)
    return out, x


def schedule64(Dw, T, L, n, real):
    """Steps of while (t <= T) t += dt with dt = 0.99 h^2 / (6 Dw), in Real."""
    t = np.float32 if real == "f32" else np.float64
    d = t(t(Dw) / t(t(L) * t(L)))
    h = t(1.0 / n)
    dt = t(0.99 * float(h) * float(h) / (6 * float(d)))
    now, k = t(0), 0
    while now <= t(T):
        now, k = t(now + dt), k + 1
    return float(d), float(dt), k


def exact_generation(case, seed):
    anat, which, rows, _ = population(case, seed)
    bpd, _, data, obs = anat[0]
    (gm, wm, csf), xs = on_grid(bpd, data, case["real"])
    pw, pg = voted(gm, wm, csf)
    tissue = torch.where(pw + pg > 0, gm + wm, 0.0)
    x = torch.from_numpy(xs).to(DEV)
    out = np.zeros((len(rows), 4))
    for i, (Dw, rho, T, *c) in enumerate(rows):
        d, dt, steps = schedule64(Dw, T, 0.1 * max(data[0].shape), 8 * bpd, case["real"])
        r = ((x[None, None, :] - c[0]) ** 2 + (x[None, :, None] - c[1]) ** 2 + (x[:, None, None] - c[2]) ** 2).sqrt()
        psi = (r - 0.005) * 64
        edge = torch.where((psi.abs() <= 1) & (tissue > 0), 0.5 * (1 - psi - torch.sin(math.pi * psi) / math.pi), 0.0)
        u = torch.where((psi < -1) & (tissue > 0.001), 1.0, edge)
        m = Model(pw, pg, d, rho, 8 * bpd)
        for _ in range(steps):
            u = m.step(u, dt)
        out[i] = likelihood64(u, obs, 3)[0][:4]
    return out


def exact_gradients(case, seed):
    anat, which, rows, steps = population(case, seed)
    loss, grad = np.zeros((len(rows), 4)), np.zeros((len(rows), 6))
    for i, (Dw, rho, T, *c) in enumerate(rows):
        bpd, _, data, obs = anat[which[i]]
        pw, pg = voted(*on_grid(bpd, data, case["real"])[0])
        m = Model(pw, pg, Dw, rho, 8 * bpd)
        loss[i], grad[i] = adjoint64(m, gaussian(8 * bpd, c, pw, pg), int(steps[i]), T, obs, c, Dw)
    return {"loss": loss, **{"grad%d" % q: np.ascontiguousarray(grad[:, q]) for q in range(6)}}


class Tree:
    """Where each block of a multi-level grid is, and its ghost cells' terms."""

    TAPS = ((-1, -1 / 16), (0, 9 / 16), (1, 9 / 16), (2, -1 / 16))  # of an odd point, from (q - 1) / 2

    def __init__(self, rows):
        self.rows = rows
        self.maps = {}
        inside = None
        for L in range(int(rows[:, 0].max()), -1, -1):
            m = np.full((1 << L,) * 3, -1, np.int64)  # -1: inside a coarser leaf
            if inside is not None:
                m[inside.reshape(1 << L, 2, 1 << L, 2, 1 << L, 2).any((1, 3, 5))] = -2
            s = np.nonzero(rows[:, 0] == L)[0]
            m[rows[s, 3], rows[s, 2], rows[s, 1]] = s
            self.maps[L] = m
            inside = m != -1

    def block(self, L, q):
        return self.maps[L][q[:, 2] >> 3, q[:, 1] >> 3, q[:, 0] >> 3] if L in self.maps else np.full(len(q), -1)

    def terms(self, L, q, to, w, out):
        """Appends (to, cell, weight) of the lattice points q of level L."""
        if not len(q):
            return
        q = q & ((8 << L) - 1)
        b = self.block(L, q)
        k = b >= 0
        out.append((to[k], b[k] * 512 + (q[k, 0] & 7) + 8 * (q[k, 1] & 7) + 64 * (q[k, 2] & 7), w[k]))
        k = b == -2
        self.terms(L + 1, 2 * q[k], to[k], w[k], out)
        k = b == -1
        q, to, w = q[k], to[k], w[k]
        for a in range(3):  # one axis after the other: even points keep theirs, odd ones get four
            odd = (q[:, a] & 1) == 1
            even = q[~odd].copy()
            even[:, a] >>= 1
            parts = [(even, to[~odd], w[~odd])]
            for o, f in self.TAPS:
                p = q[odd].copy()
                p[:, a] = (p[:, a] >> 1) + o
                parts.append((p, to[odd], w[odd] * f))
            q, to, w = (np.concatenate(v) for v in zip(*parts))
        self.terms(L - 1, q, to, w, out)

    def faces(self):
        """Index of the six face halos of every block into [cells, ghosts], and the ghosts' terms."""
        v, u = (a.reshape(-1) for a in np.meshgrid(np.arange(8), np.arange(8), indexing="ij"))
        e = np.zeros_like(u)
        at = [(e - 1, u, v), (e + 8, u, v), (u, e - 1, v), (u, e + 8, v), (u, v, e - 1), (u, v, e + 8)]
        nb = len(self.rows)
        idx = np.zeros((nb, 6, 64), np.int64)
        out, n = [], 0
        for L in self.maps:
            s = np.nonzero(self.rows[:, 0] == L)[0]
            if not len(s):
                continue
            for f in range(6):
                q = (8 * self.rows[s, 1:].astype(np.int64)[:, None, :] + np.stack(at[f], 1)[None]) & ((8 << L) - 1)
                b = self.block(L, q.reshape(-1, 3)).reshape(len(s), 64)
                same = b[:, 0] >= 0
                cell = (q[..., 0] & 7) + 8 * (q[..., 1] & 7) + 64 * (q[..., 2] & 7)
                idx[s[same], f] = b[same] * 512 + cell[same]
                g = n + np.arange(64 * int((~same).sum()))
                idx[s[~same], f] = nb * 512 + g.reshape(-1, 64)
                self.terms(L, q[~same].reshape(-1, 3), g, np.ones(len(g)), out)
                n += len(g)
        return idx, [np.concatenate(a) for a in zip(*out)], n


def exact_adaptive_steps(case, seed):
    rows, fields, Dw, rho, dt = adapted(case, seed)
    idx, (to, cell, w), ng = Tree(rows).faces()
    to, cell, w, idx = (torch.from_numpy(a).to(DEV) for a in (to, cell, w, idx))
    nb = len(rows)

    def halo(f):
        """(6 neighbours of every cell): (6, nb, z, y, x)."""
        g = torch.zeros(ng, device=DEV, dtype=F64).index_add_(0, to, f.reshape(-1)[cell] * w)
        h = torch.cat([f.reshape(-1), g])[idx].reshape(nb, 6, 8, 8)
        return [torch.cat([h[:, 0, :, :, None], f[..., :-1]], 3), torch.cat([f[..., 1:], h[:, 1, :, :, None]], 3),
                torch.cat([h[:, 2, :, None, :], f[:, :, :-1]], 2), torch.cat([f[:, :, 1:], h[:, 3, :, None, :]], 2),
                torch.cat([h[:, 4, None], f[:, :-1]], 1), torch.cat([f[:, 1:], h[:, 5, None]], 1)]

    u, pw, pg = (torch.from_numpy(a).to(DEV, F64).reshape(nb, 8, 8, 8) for a in fields[:3])
    nw, ng_ = halo(pw), halo(pg)
    D = [harmonic(a * Dw + b * 0.1 * Dw, pw * Dw + pg * 0.1 * Dw) for a, b in zip(nw, ng_)]
    t = [a + b for a, b in zip(nw, ng_)]
    ih2 = torch.exp2(2 * torch.from_numpy(rows[:, 0]).to(DEV, F64) + 6).reshape(nb, 1, 1, 1)
    for _ in range(case["steps"]):
        un = halo(u)
        d = [D[i] * (((un[i ^ 1] + t[i ^ 1]) < 0.1).to(F64) + 1) for i in range(6)]
        f = sum(d[i] * un[i] for i in range(6)) - sum(d) * u
        u = (u + dt * torch.where(u + pw + pg > 0, ih2 * f + rho * u * (1 - u), 0.0)).clamp(0, 1)
    return u


def exact(case, seed):
    kind = case["kind"]
    if kind == "adaptive_run":
        return None  # which blocks are split and merged is decided in Real
    if kind == "generation":
        return exact_generation(case, seed)
    if kind == "gradients":
        return exact_gradients(case, seed)
    if kind == "adaptive_steps":
        return exact_adaptive_steps(case, seed)
    n = case["n"]
    brain, anatomy, phi, centre = uniform(case, seed)
    u = torch.from_numpy(phi).to(DEV, F64)
    if kind == "likelihood":
        terms = likelihood64(u, observations(brain, n, seed), case["step_pet"])[0]
        return {"terms": np.array(terms[:4]), "points": terms[4]}
    Dw, rho, dt = scales(seed, n, case)
    m = Model(*voted(*(torch.from_numpy(a).to(DEV) for a in anatomy)), Dw, rho, n)
    if kind == "adjoint":
        loss, grad = adjoint64(m, u, case["steps"], case["steps"] * dt, observations(brain, n, seed), centre, Dw)
        return {"loss": np.array(loss), **{"grad%d" % q: np.array(grad[q:q + 1]) for q in range(6)}}
    for _ in range(case["steps"]):
        u = m.step(u, dt)
    return u
