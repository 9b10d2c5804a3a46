"""Timed workloads of heatsim2_amd: what its users run, through its public calls.

listed() names the workloads, draw() gives more of the same ranges, prepare()
builds what a program holds before the call (inputs made from a seed, the
plan), run() is one pass, work() what a pass cannot do without, and exact()
the same results from plain torch in float64.

Kinds of workload:
  step            one run_adi_steps call on a device field (a program's own
                  time loop: source bookkeeping, readout or control in between)
  run             run_adi_steps_many over a whole flash or heating experiment
                  with the surface history
  curved          the same under a curved top surface
  gradient        one evaluation of an inversion: per-voxel coefficients,
                  forward, misfit and backward to kz, ky, kx, rho c and the
                  flash energy
  batch_gradient  forward and backward of many uneven samples together, down
                  to the coefficients and source fields
  batch_run       their forward histories only (a parameter sweep)

Bodies ("body"): steel (one material), stack (steel over foam, a thin layer
between them), laminate (anisotropic, delaminations as thin layers).  Cells
are 0.5 mm.
"""
import math
import random

import numpy as np
import torch

import heatsim2_amd as hs

D = (5e-4, 5e-4, 5e-4)
AMBIENT = 293.0
FLASH = 1e4            # J/m^2
GRAD_DT = 2e-3
THIN = {"steel": 100.0, "stack": 250.0, "laminate": 100.0}
# (kz, ky, kx, rho, c) of each body's materials
MATERIALS = {
    "steel": [(50.0, 50.0, 50.0, 7850.0, 470.0)],
    "stack": [(50.0, 50.0, 50.0, 7850.0, 470.0), (0.03, 0.03, 0.03, 30.0, 1500.0)],
    "laminate": [(0.6, 5.0, 5.0, 1550.0, 1200.0)],
}


def listed():
    return [
        # the CPU reference workload's cube: a call per step, where latency is all
        dict(name="cube_step", kind="step", body="steel", nz=40, ny=40, nx=40, dt=1e-3),
        # the same cube, the whole 200-step flash experiment in one call
        dict(name="cube_run", kind="run", body="steel", nz=40, ny=40, nx=40, dt=1e-3, steps=200,
             source="flash"),
        # an ordinary plate, a call per step
        dict(name="stack_step", kind="step", body="stack", nz=100, ny=200, nx=300, dt=5e-4),
        # the 256^3 two-layer stack
        dict(name="stack_256_run", kind="run", body="stack", nz=256, ny=256, nx=256, dt=5e-4,
             steps=20, source="flash"),
        # the largest single-GPU laminate
        dict(name="laminate_512_run", kind="run", body="laminate", nz=128, ny=512, nx=512,
             dt=2e-3, steps=10, source="flash"),
        # sizes as they come from a measured specimen: odd on every axis
        dict(name="laminate_ragged_run", kind="run", body="laminate", nz=61, ny=149, nx=203,
             dt=2e-3, steps=40, source="flash"),
        # long-step heating: a source on every step, strongly coupled lines
        dict(name="steel_heated_run", kind="run", body="steel", nz=96, ny=160, nx=224, dt=5e-2,
             steps=20, source="heat"),
        # a curved laminate
        dict(name="curved_run", kind="curved", body="laminate", nz=48, ny=96, nx=120, dt=2e-3,
             steps=40, source="flash"),
        # the single-instance inversion: 500 steps, checkpoints every 50
        dict(name="gradient_laminate", kind="gradient", nz=64, ny=128, nx=128, steps=500,
             every=50, cooled=False),
        # a small odd specimen on a cooled base
        dict(name="gradient_ragged", kind="gradient", nz=29, ny=45, nx=51, steps=100, every=20,
             cooled=True),
        # uneven samples of 32 to 128 cells per axis, inverted together
        dict(name="batch_gradient", kind="batch_gradient", count=24, lo=32, hi=128, smin=40,
             smax=160, every=20, mix=6),
        # their histories alone, over many parameter sets
        dict(name="batch_run", kind="batch_run", count=24, lo=32, hi=128, smin=40, smax=160,
             every=20, mix=7),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def _axes(rng, lo, hi, most):
    while True:
        s = [_log_int(rng, lo, hi) for _ in range(3)]
        if s[0] * s[1] * s[2] <= most:
            return s


def draw(rng):
    kind = rng.choice(("step", "run", "run", "run", "curved", "gradient", "batch_gradient",
                       "batch_run"))
    if kind in ("step", "run", "curved"):
        nz, ny, nx = _axes(rng, 24, 512, 33554432 if kind != "curved" else 2000000)
        body = "laminate" if kind == "curved" else rng.choice(("steel", "stack", "laminate"))
        c = dict(kind=kind, body=body, nz=nz, ny=ny, nx=nx,
                 dt=round(math.exp(rng.uniform(math.log(5e-4), math.log(5e-2))), 6))
        if kind != "step":
            most = max(5, min(200, 300000000 // (nz * ny * nx)))
            c["steps"] = _log_int(rng, 5, most)
            c["source"] = rng.choice(("flash", "flash", "heat"))
        return c
    if kind == "gradient":
        nz, ny, nx = _axes(rng, 24, 160, 1000000)
        return dict(kind=kind, nz=nz, ny=ny, nx=nx, steps=_log_int(rng, 40, 400),
                    every=rng.choice((10, 20, 25, 50)), cooled=rng.random() < 0.3)
    smin = _log_int(rng, 20, 60)
    return dict(kind=kind, count=rng.randint(8, 24), lo=32, hi=rng.randint(64, 128), smin=smin,
                smax=smin + rng.randint(20, 80), every=rng.choice((10, 20, 25)),
                mix=rng.randint(0, 1 << 20))


# ---------------------------------------------------------------- inputs
def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _shape(case):
    return case["nz"], case["ny"], case["nx"]


def _maps(shape, body, rng):
    """uint8 maps: material, z / y / x faces (0 conducting, 1 insulating,
    2 thin layer), volumetric class (1 on the top layer)."""
    nz, ny, nx = shape
    mat, bz, by, bx, vol = hs.zero_elements(nz, ny, nx)
    bz[0] = bz[-1] = 1
    by[:, 0] = by[:, -1] = 1
    bx[:, :, 0] = bx[:, :, -1] = 1
    vol[0] = 1
    if body == "stack":
        top = max(1, nz // 8)
        mat[top:] = 1
        bz[top] = 2
    elif body == "laminate":
        for _ in range(int(rng.integers(1, 9))):
            sy, sx = (int(rng.integers(max(1, n // 10), max(2, n // 3))) for n in (ny, nx))
            y0, x0 = int(rng.integers(0, ny - sy + 1)), int(rng.integers(0, nx - sx + 1))
            bz[int(rng.integers(1, nz)), y0:y0 + sy, x0:x0 + sx] = 2
    return mat, bz, by, bx, vol


def _curvatures(shape, rng):
    """Top-surface curvatures (1/m), edges staying positive over the depth."""
    nz, ny, nx = shape
    most = min(15.0, 0.4 / (nz * D[0]))
    j, i = np.linspace(-1, 1, ny)[:, None], np.linspace(-1, 1, nx)[None, :]
    a, b = rng.uniform(0.3, 1.0, 2)
    return (most * a * np.cos(1.5 * j) * np.ones_like(i), most * b * np.cos(1.5 * i) * np.ones_like(j))


def _field0(shape, warm, gen):
    """A field as it stands at the call: ambient with 0.2 K of unevenness,
    plus what an earlier flash left under the surface when `warm`."""
    T = AMBIENT + 0.2 * torch.rand(shape, dtype=torch.float64, device=_dev(), generator=gen)
    if warm:
        z = torch.arange(shape[0], dtype=torch.float64, device=_dev()) * D[0]
        T += (5.0 * torch.exp(-z / 4e-3))[:, None, None]
    return T


def _smooth(shape, gen):
    """A smooth random field in about [-1, 1] (correlation of some 8 cells)."""
    coarse = [max(2, n // 8) for n in shape]
    g = torch.rand([1, 1] + coarse, dtype=torch.float64, device=_dev(), generator=gen) * 2 - 1
    return torch.nn.functional.interpolate(g, size=list(shape), mode="trilinear",
                                           align_corners=True)[0, 0].contiguous()


def _volumetric(case, E):
    if case.get("source") == "flash":
        return [(hs.NO_SOURCE,), (hs.IMPULSE_SOURCE, 0.0, E / D[0])]
    if case.get("source") == "heat":  # on throughout
        return [(hs.NO_SOURCE,),
                (hs.STEPPED_SOURCE, 0.0, case["dt"] * (case["steps"] + 1), E / (0.5 * D[0]))]
    return [(hs.NO_SOURCE,), (hs.IMPULSE_SOURCE, -1.0, E / D[0])]  # fired before


def _energy(rng):
    return FLASH * (1.0 + 0.05 * rng.uniform(-1.0, 1.0))


def _cooling(E, k, rhoc, nsteps, dt, shape):
    """A plain half-space's surface cooling after a flash, (nsteps, 1, 1)."""
    t = (torch.arange(nsteps, dtype=torch.float64, device=_dev()) + 1.0) * dt
    return (E / torch.sqrt(math.pi * k * rhoc * t))[:, None, None]


def _samples(case):
    """Sizes, step counts and materials of a batch's samples."""
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["count"]):
        shape = tuple(r.randint(case["lo"], case["hi"]) for _ in range(3))
        lk = [math.exp(r.uniform(math.log(0.1), math.log(60.0))) for _ in range(3)]
        if r.random() < 0.5:
            lk = [lk[0]] * 3
        out.append(dict(shape=shape, steps=r.randint(case["smin"], case["smax"]), k=lk,
                        rhoc=math.exp(r.uniform(math.log(1e5), math.log(5e6)))))
    return out


def _conductance(k, face, d, axis, fixed=None, h=100.0):
    """Minus-face conductance per volume along `axis` (0 on the first face):
    (k_m + k_p) / (2 d^2), a fixed neighbour's k replaced by the cell's own;
    h / d across a thin layer; 0 across an insulating face."""
    n = k.shape[axis]
    km, kp = k.narrow(axis, 0, n - 1), k.narrow(axis, 1, n - 1)
    if fixed is not None:
        fm, fp = fixed.narrow(axis, 0, n - 1), fixed.narrow(axis, 1, n - 1)
        km, kp = torch.where(fm, kp, km), torch.where(fp, km, kp)
    b = torch.as_tensor(face, device=k.device).narrow(axis, 1, n - 1)
    g = torch.where(b == 0, (km + kp) / (2.0 * d * d),
                    torch.where(b == 2, torch.full_like(km, h / d), torch.zeros_like(km)))
    if fixed is not None:
        g = torch.where(fm & fp, torch.zeros_like(g), g)
    return torch.cat((torch.zeros_like(k.narrow(axis, 0, 1)), g), axis)


def _batch_inputs(case, seed):
    """Flat coefficient vectors (samples one after another), per-sample
    initial fields, flash fields and observations."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=_dev()).manual_seed(seed)
    parts = {n: [] for n in ("M", "gz", "gy", "gx", "src")}
    w, T0, obs = [], [], []
    samples = _samples(case)
    for s in samples:
        sh = s["shape"]
        _, bz, by, bx, _ = _maps(sh, "laminate", rng)
        E = _energy(rng)
        k = [kk * (1.0 + 0.2 * _smooth(sh, gen)) for kk in s["k"]]
        rhoc = s["rhoc"] * (1.0 + 0.1 * _smooth(sh, gen))
        parts["M"].append(rhoc / GRAD_DT)
        for a, (n, f) in enumerate((("gz", bz), ("gy", by), ("gx", bx))):
            parts[n].append(_conductance(k[a], f, D[a], a))
        S = torch.zeros(sh, dtype=torch.float64, device=_dev())
        S[0] = E / (D[0] * GRAD_DT)
        parts["src"].append(S)
        w.append(torch.ones(sh, dtype=torch.uint8, device=_dev()))
        T0.append(torch.zeros(sh, dtype=torch.float64, device=_dev()))
        noise = torch.randn((s["steps"],) + sh[1:], dtype=torch.float64, device=_dev(),
                            generator=gen)
        obs.append(_cooling(E, s["k"][0], s["rhoc"], s["steps"], GRAD_DT, sh) + 0.01 * noise)
    flat = {n: torch.cat([p.reshape(-1) for p in v]) for n, v in parts.items()}
    return samples, flat, w, T0, obs


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=_dev()).manual_seed(seed)
    kind = case["kind"]
    if kind in ("step", "run", "curved"):
        shape = _shape(case)
        body = case["body"]
        maps = _maps(shape, body, rng)
        E = _energy(rng)
        mats = []
        for kz, ky, kx, rho, c in MATERIALS[body]:
            k = np.diag([kz, ky, kx]) if body == "laminate" else kz
            mats.append((hs.TEMPERATURE_COMPUTE, k, rho, c))
        law = hs.boundary_conducting_anisotropic if body == "laminate" else hs.boundary_conducting
        bnds = [(law,), (hs.boundary_insulating,),
                (hs.boundary_thininsulatinglayer, THIN[body])]
        vol = _volumetric(case, E)
        curv = _curvatures(shape, rng) if kind == "curved" else (None, None)
        P, S = hs.setup(D[0] / 2, D[1] / 2, D[2] / 2, D[0], D[1], D[2], *shape, case["dt"], mats,
                        bnds, vol, *maps, *curv)
        return dict(kind=kind, P=P, S=S, dt=case["dt"], steps=case.get("steps"), vol=vol,
                    vmap=maps[4], maps=maps, E=E, curv=curv,
                    T=_field0(shape, kind == "step", gen))
    if kind == "gradient":
        shape = _shape(case)
        _, bz, by, bx, _ = _maps(shape, "laminate", rng)
        kz, ky, kx, rho, c = MATERIALS["laminate"][0]
        E = _energy(rng)
        p = dict(kz=kz * (1.0 + 0.3 * _smooth(shape, gen)),
                 ky=ky * (1.0 + 0.1 * _smooth(shape, gen)),
                 kx=kx * (1.0 + 0.1 * _smooth(shape, gen)),
                 rhoc=rho * c * (1.0 + 0.05 * _smooth(shape, gen)),
                 E=torch.tensor(E, dtype=torch.float64, device=_dev()))
        fixed = None
        if case["cooled"]:
            fixed = torch.zeros(shape, dtype=torch.bool, device=_dev())
            fixed[-1] = True
        mask = torch.zeros(shape, dtype=torch.float64, device=_dev())
        mask[0] = 1.0
        noise = torch.randn((case["steps"],) + shape[1:], dtype=torch.float64, device=_dev(),
                            generator=gen)
        return dict(kind=kind, p={n: v.requires_grad_(True) for n, v in p.items()},
                    maps=(bz, by, bx), fixed=fixed, mask=mask, steps=case["steps"],
                    every=case["every"], T0=torch.zeros(shape, dtype=torch.float64, device=_dev()),
                    obs=_cooling(E, kz, rho * c, case["steps"], GRAD_DT, shape) + 0.01 * noise,
                    bnds=((hs.boundary_conducting_anisotropic,), (hs.boundary_insulating,),
                          (hs.boundary_thininsulatinglayer, THIN["laminate"])),
                    plan=hs.adjoint.GradPlan(shape, D, GRAD_DT))
    samples, flat, w, T0, obs = _batch_inputs(case, seed)
    gb = hs.batch.GradBatch([s["shape"] for s in samples], D[0], [s["steps"] for s in samples],
                            [0] * len(samples), ckpt_every=case["every"])
    if kind == "batch_gradient":
        flat = {n: v.requires_grad_(True) for n, v in flat.items()}
    return dict(kind=kind, samples=samples, flat=flat, w=w, T0=T0, obs=obs, gb=gb)


# ------------------------------------------------------------------ a pass
def _split(flat, samples):
    parts = torch.split(flat, [int(np.prod(s["shape"])) for s in samples])
    return [p.view(s["shape"]) for p, s in zip(parts, samples)]


def run(s):
    kind = s["kind"]
    if kind == "step":
        return hs.run_adi_steps(s["P"], s["S"], 0.0, s["dt"], s["T"], s["vmap"], s["vol"])
    if kind in ("run", "curved"):
        return hs.run_adi_steps_many(s["P"], 0.0, s["dt"], s["steps"], s["T"], s["vmap"],
                                     s["vol"], surface_history=True)
    if kind == "gradient":
        p = s["p"]
        coef = hs.adjoint.per_voxel_coefficients(p["kz"], p["ky"], p["kx"], p["rhoc"], GRAD_DT, D,
                                                 s["bnds"], *s["maps"], fixed=s["fixed"])
        hist = hs.adjoint.surface_history(s["plan"], coef, s["T0"], s["steps"],
                                          sources=[(0, p["E"] * s["mask"] / (D[0] * GRAD_DT))],
                                          ckpt_every=s["every"])
        loss = ((hist - s["obs"]) ** 2).sum()
        names = ("kz", "ky", "kx", "rhoc", "E")
        grads = torch.autograd.grad(loss, [p[n] for n in names])
        return dict(zip(names, grads), loss=loss.detach(), hist=hist.detach())
    fields = {n: _split(v, s["samples"]) for n, v in s["flat"].items()}
    coefs = [dict(M=fields["M"][i], w=s["w"][i], gz=fields["gz"][i], gy=fields["gy"][i],
                  gx=fields["gx"][i]) for i in range(len(s["w"]))]
    if kind == "batch_run":
        return s["gb"].run(coefs, s["T0"], fields["src"])
    hists = s["gb"].surface_history(coefs, s["T0"], fields["src"])
    loss = sum(((h - o) ** 2).sum() for h, o in zip(hists, s["obs"]))
    names = ("M", "gz", "gy", "gx", "src")
    grads = torch.autograd.grad(loss, [s["flat"][n] for n in names])
    return dict(zip(names, grads), loss=loss.detach(), hists=[h.detach() for h in hists])


def work(case):
    """Bytes and operations of one pass.  A step reads and writes the field
    once and solves three lines per cell (about 60 operations); per-voxel
    coefficients (M, three conductances, the row flag) are read with it.  A
    gradient also walks the steps backwards, with the states of each step and
    the four gradient fields read and written."""
    kind = case["kind"]
    if kind.startswith("batch"):
        insts = _samples(case)
    else:
        insts = [dict(shape=_shape(case), steps=case.get("steps", 1))]
    nbytes = flops = 0.0
    for s in insts:
        n = float(np.prod(s["shape"]))
        top = float(s["shape"][1] * s["shape"][2])
        coef = {"step": 1.0, "run": 1.0, "curved": 57.0}.get(kind, 33.0)
        per = 16.0 + coef
        ops = 60.0
        if "gradient" in kind:
            per += 16.0 + coef + 24.0 + 64.0
            ops += 200.0
        nbytes += s["steps"] * (n * per + (8.0 * top if kind != "step" else 0.0))
        flops += s["steps"] * n * ops
    return {"bytes": nbytes, "flops": flops}


# --------------------------------------------------------- plain float64
def _factor(a, b, c):
    """Thomas factors of the systems a x[t-1] + b x[t] + c x[t+1] = r along
    the first axis, as per-row lists (1/pivot, a/pivot, c/pivot)."""
    inv, low, up = [], [], []
    for t in range(len(b)):
        d = b[t] - a[t] * up[-1] if t else b[t]
        inv.append(1.0 / d)
        low.append(a[t] * inv[-1])
        up.append(c[t] * inv[-1])
    return torch.stack(inv), low, up


def _solve(factors, r):
    inv, low, up = factors
    y = list((r * inv).unbind(0))
    for t in range(1, len(y)):
        y[t] = torch.addcmul(y[t], low[t], y[t - 1], value=-1)
    for t in range(len(y) - 2, -1, -1):
        y[t] = torch.addcmul(y[t], up[t], y[t + 1], value=-1)
    return torch.stack(y)


class _Plain(object):
    """The Douglas step x, y, z in float64: M per cell, minus- and plus-face
    conductances gm[a], gp[a] of array axes z, y, x (0 on outer faces and in
    fixed rows)."""

    def __init__(self, M, gm, gp):
        self.M, self.gm, self.gp = M, gm, gp
        self.f = []
        for a in range(3):
            lo, hi = (-0.5 * g.movedim(a, 0) for g in (gm[a], gp[a]))
            self.f.append(_factor(lo, M.movedim(a, 0) - lo - hi, hi))

    def lap(self, a, T):
        d = torch.diff(T, dim=a)
        z = torch.zeros_like(T.narrow(a, 0, 1))
        return self.gp[a] * torch.cat((d, z), a) - self.gm[a] * torch.cat((z, d), a)

    def solve(self, a, r):
        return _solve(self.f[a], r.movedim(a, 0)).movedim(0, a)

    def step(self, T, S=None):
        lz, ly, lx = (self.lap(a, T) for a in range(3))
        r = self.M * T + 0.5 * lx + ly + lz
        if S is not None:
            r = r + S
        X = self.solve(2, r)
        X = self.solve(1, self.M * X - 0.5 * ly)
        return self.solve(0, self.M * X - 0.5 * lz)


def _readout(T):
    return T[0] - 0.3125 * (T[1] - T[0])


def _plus(g, axis):
    n = g.shape[axis]
    return torch.cat((g.narrow(axis, 1, n - 1), torch.zeros_like(g.narrow(axis, 0, 1))), axis)


def _plain_body(case, maps, curv):
    body = case["body"]
    mat = torch.as_tensor(maps[0], device=_dev()).long()
    tab = torch.tensor(MATERIALS[body], dtype=torch.float64, device=_dev())
    M = (tab[:, 3] * tab[:, 4])[mat] / case["dt"]
    k = [tab[:, a][mat] for a in range(3)]
    gm = [_conductance(k[a], maps[1 + a], D[a], a, h=THIN[body]) for a in range(3)]
    gp = [_plus(gm[a], a) for a in range(3)]
    if curv[0] is not None:
        # a cell's faces weighed by its own areas over its own volume, the
        # conducting laws taken at its own mean spacings
        nz = case["nz"]
        q = torch.arange(nz, dtype=torch.float64, device=_dev())[:, None, None] * D[0]
        ky, kx = (torch.as_tensor(c, device=_dev())[None] for c in curv)
        yt, yb = (1 + q * ky) * D[1], (1 + (q + D[0]) * ky) * D[1]
        xt, xb = (1 + q * kx) * D[2], (1 + (q + D[0]) * kx) * D[2]
        ym, xm = (yt + yb) / 2, (xt + xb) / 2
        V = xm * ym * D[0]
        gm[0], gp[0] = gm[0] * D[0] * xt * yt / V, gp[0] * D[0] * xb * yb / V
        for a, m, area in ((1, ym, xm * D[0]), (2, xm, ym * D[0])):
            # k / d becomes k / (mean spacing); only conducting faces occur
            gm[a], gp[a] = (g * D[a] * (D[a] / m) * area / V for g in (gm[a], gp[a]))
    return _Plain(M, gm, gp)


def _exact_gradient(case, seed):
    s = prepare(case, seed)
    p = {n: v.detach().clone().requires_grad_(True) for n, v in s["p"].items()}
    small = case["steps"] * sum(_shape(case)) <= 40000  # the whole graph is kept
    with torch.set_grad_enabled(small):
        fixed = s["fixed"]
        k = [p["kz"], p["ky"], p["kx"]]
        gm = [_conductance(k[a], s["maps"][a], D[a], a, fixed) for a in range(3)]
        gp = [_plus(g, a) for a, g in enumerate(gm)]
        M = p["rhoc"] / GRAD_DT
        S = p["E"] * s["mask"] / (D[0] * GRAD_DT)
        if fixed is not None:
            gm, gp = ([torch.where(fixed, torch.zeros_like(g), g) for g in v] for v in (gm, gp))
            M = torch.where(fixed, torch.ones_like(M), M)
        plain, T, hist = _Plain(M, gm, gp), s["T0"], []
        for n in range(case["steps"]):
            T = plain.step(T, S if n == 0 else None)
            hist.append(_readout(T))
        hist = torch.stack(hist)
        loss = ((hist - s["obs"]) ** 2).sum()
    names = ("kz", "ky", "kx", "rhoc", "E")
    grads = torch.autograd.grad(loss, [p[n] for n in names]) if small else [None] * 5
    return dict(zip(names, grads), loss=loss.detach(), hist=hist.detach())


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch_gradient":
        return None
    if kind == "gradient":
        return _exact_gradient(case, seed)
    with torch.no_grad():
        if kind == "batch_run":
            samples, flat, _, T0, _ = _batch_inputs(case, seed)
            f = {n: _split(v, samples) for n, v in flat.items()}
            Ts, hists = [], []
            for i, x in enumerate(samples):
                g = [f[n][i] for n in ("gz", "gy", "gx")]
                plain = _Plain(f["M"][i], g, [_plus(v, a) for a, v in enumerate(g)])
                T, h = T0[i], []
                for n in range(x["steps"]):
                    T = plain.step(T, f["src"][i] if n == 0 else None)
                    h.append(_readout(T))
                Ts.append(T)
                hists.append(torch.stack(h))
            return Ts, hists
        s = prepare(case, seed)
        plain, T = _plain_body(case, s["maps"], s["curv"]), s["T"]
        if kind == "step":
            return plain.step(T)
        S = torch.zeros_like(T)
        flash = case["source"] == "flash"
        S[0] = s["E"] / (D[0] * case["dt"]) if flash else s["E"] / (0.5 * D[0])
        h = []
        for n in range(case["steps"]):
            T = plain.step(T, S if n == 0 or not flash else None)
            h.append(_readout(T))
        return T, torch.stack(h)
