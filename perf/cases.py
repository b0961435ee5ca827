"""Workloads whose speed and results are compared between two versions of this package.

A case is one call pattern of a program that uses ela3d_amd, at one grid:

* ``run``    a whole forward shot: create it, run its steps, read seismograms and energy;
* ``steps``  a shot that a program keeps on the GPU and advances by a block of steps,
             then reads the seismograms and energy recorded so far;
* ``look``   the same with a wavefield read back after each block (a snapshot);
* ``serve``  a server that is given a list of shots of mixed sizes and returns their
             seismograms.

Grids, media, storages and options are those of ``ela3d_amd.workloads``, of the tests and
of ``bench.py``.  The model of a grid is fixed (one survey, many shots); the seed draws
source position, frequency and receivers.  Results come back in the type that the storage
carries: float32, float64, and float16 for FP16 storage.
"""
import functools
import math

import numpy as np
import torch

import ela3d_amd as ela
from ela3d_amd import workloads

STORAGE = {"fp32": ela.STORAGE_FP32, "fp16": ela.STORAGE_FP16, "fp64": ela.STORAGE_FP64}
OUT = {"fp32": np.float32, "fp16": np.float16, "fp64": np.float64}
BYTES = {"fp32": 4, "fp16": 2, "fp64": 8}
SOURCE = {"force": ela.SRC_FORCE, "explosive": ela.SRC_EXPLOSIVE, "sigma": ela.SRC_REFERENCE_SIGMA,
          "force3": ela.SRC_FORCE3}
WAVELET = {"ricker": ela.WAVELET_RICKER, "gaussian": ela.WAVELET_GAUSSIAN, "dgaussian": ela.WAVELET_DGAUSSIAN}


def _case(name, kind, nx, ny, nz, **kw):
    """steps: steps of one pass; warm: steps a kept shot has behind it; nstep: its planned length."""
    c = dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, storage="fp32", model="layered", source="force",
             wavelet="ricker", steps=20, warm=0, nstep=0, energy=0, nrec=64, sample=1,
             free_surface=False, reference=False, tuned=False)
    c.update(kw)
    c["nstep"] = c["nstep"] or c["steps"] + c["warm"]
    return c


def listed():
    return [
        # the smallest use: two steps of a toy grid, then one field is looked at (a program
        # that steers or draws while it steps); launches and latency are all there is
        _case("look_33", "look", 33, 33, 33, model="homogeneous", steps=2, warm=100, nstep=400, nrec=9),
        # the smallest shots of the serving stream, run one by one
        _case("run_64", "run", 64, 64, 64, steps=200),
        # the homogeneous 101^3 cube with the energy summed at every step
        _case("run_cube_101", "run", 101, 101, 101, model="homogeneous", steps=300, energy=1, nrec=42),
        # land survey geometry: a free surface, sides that are no multiples of anything
        _case("run_surface_ragged", "run", 113, 97, 85, steps=200, source="explosive", energy=10,
              free_surface=True),
        # the reference program's own choices (its quirks, sigma source, derivative of a
        # Gaussian) in double precision
        _case("run_reference_fp64", "run", 81, 61, 75, storage="fp64", model="homogeneous", source="sigma",
              wavelet="dgaussian", steps=150, reference=True),
        # the MATLAB anticline at its own size
        _case("steps_anticline_201", "steps", 201, 201, 201, model="anticline", source="explosive", steps=40,
              warm=100, nstep=2000, energy=10, nrec=256, sample=5),
        # the layered anticline, 48 million cells with 401-cell rows, in both storages
        _case("steps_layered", "steps", 401, 401, 301, source="explosive", steps=20, warm=100, nstep=2000,
              energy=10, nrec=256, sample=5),
        _case("steps_layered_fp16", "steps", 401, 401, 301, storage="fp16", source="explosive", steps=20,
              warm=100, nstep=2000, nrec=256, sample=5),
        # a program that runs many shots on the classic 101 x 641 x 640 grid tunes it once
        _case("steps_classic_tuned", "steps", 101, 641, 640, model="homogeneous", steps=40, warm=100, nstep=2500,
              energy=10, nrec=65, sample=5, tuned=True),
        # a reference run in double precision at a size that fills the GPU
        _case("steps_fp64", "steps", 192, 200, 188, storage="fp64", model="homogeneous", steps=20, warm=80,
              nstep=2000, energy=10, nrec=200, sample=5),
        # the largest: 86 million cells, wide rows, rigid model of one medium
        _case("steps_large", "steps", 480, 500, 360, model="homogeneous", source="force3", steps=20, warm=60,
              nstep=2000, nrec=256, sample=5),
        # serving: shots of mixed sizes submitted together, results collected in order
        _case("serve_mix", "serve", 64, 256, 10, steps=120),
    ]


def draw(rng):
    """One more case.  The sides of a grid are drawn over the logarithm of their range and
    differ; a ``serve`` case holds its smallest edge, largest edge and number of shots."""
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["look", "run", "run", "steps", "steps", "steps", "serve"])
    if kind == "serve":
        lo = side(48, 80)
        c = _case("", kind, lo, lo + side(30, 150), rng.randint(4, 10), steps=rng.randint(60, 120))
    else:
        hi = {"look": 60, "run": 150, "steps": 420}[kind]
        lo = {"look": 30, "run": 48, "steps": 100}[kind]
        nx, ny, nz = side(lo, hi), side(lo, hi), side(lo, hi)
        storage = rng.choice(["fp32", "fp32", "fp32", "fp16", "fp64"])
        source = rng.choice(["force", "explosive", "force3", "sigma"])
        c = _case("", kind, nx, ny, nz, storage=storage, source=source,
                  model=rng.choice(["homogeneous", "layered"]),
                  wavelet="ricker" if storage == "fp16" else rng.choice(["ricker", "ricker", "dgaussian"]),
                  energy=0 if storage == "fp16" else rng.choice([0, 1, 10]),
                  free_surface=rng.random() < 0.25,
                  nrec=rng.randint(4, 256), sample={"look": 1, "run": rng.choice([1, 2]), "steps": 5}[kind],
                  steps={"look": rng.randint(1, 4), "run": rng.randint(100, 200), "steps": rng.randint(10, 20)}[kind],
                  warm={"look": 100, "run": 0, "steps": 80}[kind])
        c["nstep"] = c["steps"] + c["warm"] if kind == "run" else 2000
    del c["name"]
    return c


@functools.lru_cache(maxsize=6)
def _model(kind, nx, ny, nz):
    """(cp, cs, rho, largest cp) of a grid."""
    if kind == "anticline":
        m = ela.anticline_model(nx)
        return m + (float(m[0].max()),)
    if kind == "layered":
        depth = nz * 10.0
        return ela.layered_model(nx, ny, nz, 10.0, bump_amp=0.15 * depth, bump_width=0.3 * depth)
    return ela.homogeneous_model(nx, ny, nz, workloads.CP, workloads.CS, workloads.RHO) + (workloads.CP,)


def _receivers(rng, dims, src, n):
    """Half the stations within 20 cells of the source, the others anywhere inside the layers."""
    dims, src = np.asarray(dims), np.asarray(src)
    far = rng.integers(11, dims - 11, size=(n - n // 2, 3))
    near = np.clip(src + rng.integers(-20, 21, size=(n // 2, 3)), 1, dims - 2)
    return np.concatenate([near, far]).astype(np.int32)


def _shot(case, seed):
    """(Config, model) of the case's shot."""
    rng = np.random.default_rng([seed, 17])
    nx, ny, nz = dims = case["nx"], case["ny"], case["nz"]
    cp, cs, rho, vmax = _model(case["model"], nx, ny, nz)
    src = [int(rng.integers(13, n - 13)) for n in dims]
    f0 = float(rng.uniform(18.0, 24.0))
    kw = dict(receivers=_receivers(rng, dims, src, case["nrec"]), energy_every=case["energy"],
              sample_every=case["sample"], storage=STORAGE[case["storage"]], free_surface=case["free_surface"], vpml=vmax,
              src_kind=SOURCE[case["source"]], wavelet=WAVELET[case["wavelet"]], isrc=src[0], jsrc=src[1],
              ksrc=src[2], angle_force=float(rng.uniform(0.0, 90.0)),
              # amplitudes whose samples float16 holds without overflow (stress sources move the ground more)
              factor=1e7 if case["storage"] != "fp16" else 1e2 if case["source"] in ("sigma", "explosive") else 1e9)
    dt = ela.courant_dt(10.0, vmax, 0.5)
    if case["reference"]:
        return ela.Config.from_reference(nx, ny, nz, 10.0, dt, case["nstep"], f0=f0, **kw), (cp, cs, rho)
    cfg = ela.Config(nx=nx, ny=ny, nz=nz, dt=dt, nstep=case["nstep"], f0=f0, **kw)
    return cfg, (cp, cs, rho)


def _serve_shots(case, seed):
    """The shots of a ``serve`` case: edges from the smallest to the largest, smaller ones more often."""
    rng = np.random.default_rng([seed, 29])
    out = []
    for q in range(case["nz"]):
        n = int(round(case["nx"] * (case["ny"] / case["nx"]) ** ((q / max(1, case["nz"] - 1)) ** 1.5)))
        cp, cs, rho, vmax = _model("layered" if q % 2 else "homogeneous", n, n, n)
        src = [int(rng.integers(13, n - 13)) for _ in range(3)]
        cfg = ela.Config(nx=n, ny=n, nz=n, dt=ela.courant_dt(10.0, vmax, 0.5),
                         nstep=case["steps"] * (10 - q % 4) // 10, f0=float(rng.uniform(18.0, 24.0)),
                         vpml=vmax, isrc=src[0], jsrc=src[1], ksrc=src[2],
                         receivers=_receivers(rng, (n, n, n), src, case["nrec"]))
        out.append((cfg, (cp, cs, rho)))
    return out


_TUNED = set()


def prepare(case, seed):
    if case["kind"] == "serve":
        return {"case": case, "server": ela.Server(), "shots": _serve_shots(case, seed)}
    cfg, model = _shot(case, seed)
    if case["tuned"] and (cfg.nx, cfg.ny, cfg.nz) not in _TUNED:  # once a program
        ela.autotune(cfg, model)
        _TUNED.add((cfg.nx, cfg.ny, cfg.nz))
    state = {"case": case, "cfg": cfg, "model": model}
    if case["kind"] != "run":
        state["shot"] = ela.Shot(cfg, *model)
        state["shot"].step(case["warm"])
        state["shot"].sync()
    return state


def run(state):
    case = state["case"]
    kind, as_ = case["kind"], OUT[case["storage"]]
    if kind == "serve":
        srv = state["server"]
        tickets = [srv.submit(cfg, *model) for cfg, model in state["shots"]]
        return [srv.result(t)[0].astype(np.float32) for t in tickets]
    if kind == "run":
        with ela.Shot(state["cfg"], *state["model"]) as shot:
            shot.run()
            return {"seismograms": shot.seismograms().astype(as_), "energy": shot.energy().astype(as_)}
    shot = state["shot"]
    shot.step(case["steps"])
    shot.sync()
    if kind == "look":
        return {"vz": shot.snapshot(2).astype(as_)}
    return {"seismograms": shot.seismograms().astype(as_), "energy": shot.energy().astype(as_)}


def work(case):
    """A step reads and writes nine fields and reads three model arrays once; where absorbing
    layers lie, it also reads and writes their memory variables (six along each axis)."""
    def step(nx, ny, nz, e, fs):
        w = 21
        pml = 6.0 * (w * ny * nz + w * nx * nz + (w - (10 if fs else 0)) * nx * ny)
        return nx * ny * nz * (18.0 * e + 12.0) + 2.0 * e * pml

    if case["kind"] == "serve":
        shots = _serve_shots(case, 1)
        by = sum(cfg.nstep * step(cfg.nx, cfg.ny, cfg.nz, 4, False) for cfg, _ in shots)
        return {"bytes": by, "flops": sum(110.0 * cfg.cells * cfg.nstep for cfg, _ in shots)}
    e = BYTES[case["storage"]]
    by = case["steps"] * step(case["nx"], case["ny"], case["nz"], e, case["free_surface"])
    return {"bytes": by, "flops": 110.0 * case["nx"] * case["ny"] * case["nz"] * case["steps"]}


# ---- the same loop in plain 64-bit torch ---------------------------------------------------


def _tables(cfg, axis):
    """a, b, K on the full grid and on the half grid of one axis."""
    n, h = ((cfg.nx, cfg.dx), (cfg.ny, cfg.dy), (cfg.nz, cfg.dz))[axis]
    quirk_x = axis == 0 and cfg.compat_flags & ela.COMPAT_XHALF_A
    quirk_z = axis == 2 and cfg.compat_flags & ela.COMPAT_ZHALF_MIN
    thick, thick_y = cfg.npoints_pml * h, cfg.npoints_pml * cfg.dy
    norm = thick_y if quirk_z else thick
    amax = cfg.alpha_max_pml if cfg.alpha_max_pml > 0 else math.pi * cfg.f0
    d0 = -(cfg.npower + 1.0) * cfg.vpml * math.log(cfg.rcoef) / (2.0 * thick)
    out = []
    for half in (False, True):
        x = h * np.arange(n) + (h / 2.0 if half else 0.0)
        low = thick - x
        if half and quirk_z:
            low = np.full(n, thick_y - (cfg.dy * (cfg.ny - 1) + cfg.dy / 2.0))
        if axis == 2 and cfg.free_surface:
            low = np.full(n, -1.0)
        high = x - ((n - 1) * h - thick)
        s = np.where(high >= 0.0, high / (norm if half else thick), np.where(low >= 0.0, low / norm, -1.0))
        on, s = s >= 0.0, np.maximum(s, 0.0)
        d = np.where(on, d0 * s ** cfg.npower, 0.0)
        k = np.where(on, 1.0 + (cfg.k_max_pml - 1.0) * s ** cfg.npower, 1.0)
        al = np.maximum(np.where(on, amax * (1.0 - s) + 0.1 * amax, 0.0), 0.0)
        b = np.exp(-(d / k + al) * cfg.dt)
        big = np.abs(d) > 1e-6
        a = np.where(big, d * (b - 1.0) / np.where(big, k * (d + k * al), 1.0), 0.0)
        out.append((np.zeros(n) if half and quirk_x else a, b, k))
    return out


class _Plain:
    """The velocity-stress loop on whole arrays [z][y][x]."""

    def __init__(self, cfg, model, dev):
        self.c, self.dev = cfg, dev
        self.cp, self.cs, self.rho = (torch.as_tensor(m, device=dev).double() for m in model)
        self.f = [torch.zeros_like(self.cp) for _ in range(9)]
        self.tab = [_tables(cfg, a) for a in range(3)]
        self.mem = {}

    def pml(self, key, d, axis, half, where):
        """The C-PML recurrence of derivative d, which covers the index slices `where` (z, y, x)."""
        a, b, k = (t[where[2 - axis]] for t in self.tab[axis][half])
        on = np.flatnonzero(a != 0.0)
        if not len(on):
            return d
        cut = np.flatnonzero(np.diff(on) > 1)
        for run in np.split(on, cut + 1):
            sl = [slice(None)] * 3
            sl[2 - axis] = slice(int(run[0]), int(run[-1]) + 1)
            sl = tuple(sl)
            shape = [1, 1, 1]
            shape[2 - axis] = len(run)
            ta, tb, tk = (torch.as_tensor(t[run], device=self.dev).view(shape) for t in (a, b, k))
            m = self.mem.get((key, int(run[0])))
            m = ta * d[sl] if m is None else tb * m + ta * d[sl]
            self.mem[key, int(run[0])] = m
            d[sl] = d[sl] / tk + m
        return d

    def stress(self):
        c, (vx, vy, vz, sxx, syy, szz, sxy, sxz, syz) = self.c, self.f
        nx, ny, nz, dt = c.nx, c.ny, c.nz, c.dt
        fs = bool(c.free_surface)
        for k0, k1, surface in ((1, nz, False),) + (((0, 1, True),) if fs else ()):
            w = (slice(k0, k1), slice(1, ny), slice(0, nx - 1))
            exx = self.pml(("xx", k0), (vx[k0:k1, 1:, 1:] - vx[k0:k1, 1:, :-1]) / c.dx, 0, 1, w)
            eyy = self.pml(("yy", k0), (vy[k0:k1, 1:, :-1] - vy[k0:k1, :-1, :-1]) / c.dy, 1, 0, w)
            rho, cp, cs = self.rho[w], self.cp[w], self.cs[w]
            lam, l2m = rho * (cp * cp - 2.0 * cs * cs), rho * cp * cp
            if surface:
                ezz = -(lam / l2m) * (exx + eyy)
            else:
                ezz = self.pml(("zz", k0), (vz[1:, 1:, :-1] - vz[:-1, 1:, :-1]) / c.dz, 2, 0, w)
                szz[w] += dt * (lam * (exx + eyy) + l2m * ezz)
            sxx[w] += dt * (l2m * exx + lam * (eyy + ezz))
            syy[w] += dt * (lam * (exx + ezz) + l2m * eyy)
        w = (slice(0, nz), slice(0, ny - 1), slice(1, nx))
        vs = (self.cs[:, :-1, :-1] + self.cs[:, 1:, 1:]) / 2
        mu = (self.rho[:, :-1, :-1] + self.rho[:, 1:, 1:]) / 2 * vs * vs
        d = self.pml("yx", (vy[:, :-1, 1:] - vy[:, :-1, :-1]) / c.dx, 0, 0, w)
        sxy[w] += dt * mu * (d + self.pml("xy", (vx[:, 1:, 1:] - vx[:, :-1, 1:]) / c.dy, 1, 1, w))
        kt = nz if c.compat_flags & ela.COMPAT_GHOST else nz - 1

        def up(t):  # plane k + 1; a zero plane above the top one
            return t[1:] if kt == nz - 1 else torch.cat([t[1:], torch.zeros_like(t[:1])])

        cs_u, rho_u = up(self.cs), up(self.rho)
        w = (slice(0, kt), slice(0, ny), slice(1, nx))
        vs = (self.cs[:kt, :, :-1] + cs_u[:, :, 1:]) / 2
        mu = (self.rho[:kt, :, :-1] + rho_u[:, :, 1:]) / 2 * vs * vs
        d = self.pml("zx", (vz[:kt, :, 1:] - vz[:kt, :, :-1]) / c.dx, 0, 0, w)
        sxz[w] += dt * mu * (d + self.pml("xz", (up(vx)[:, :, 1:] - vx[:kt, :, 1:]) / c.dz, 2, 1, w))
        w = (slice(0, kt), slice(0, ny - 1), slice(0, nx))
        vs = (self.cs[:kt, 1:] + cs_u[:, :-1]) / 2
        mu = (self.rho[:kt, 1:] + rho_u[:, :-1]) / 2 * vs * vs
        d = self.pml("zy", (vz[:kt, 1:] - vz[:kt, :-1]) / c.dy, 1, 1, w)
        syz[w] += dt * mu * (d + self.pml("yz", (up(vy)[:, :-1] - vy[:kt, :-1]) / c.dz, 2, 1, w))

    def velocity(self):
        c, rho, (vx, vy, vz, sxx, syy, szz, sxy, sxz, syz) = self.c, self.rho, self.f
        nx, ny, nz, dt = c.nx, c.ny, c.nz, c.dt
        k0 = 0 if c.free_surface else 1  # a free surface moves plane 0 too, by the stress image below it
        w = (slice(k0, nz), slice(1, ny), slice(1, nx))
        below = torch.cat([-sxz[:1], sxz[:-1]])[k0:]
        d = self.pml("sxx", (sxx[k0:, 1:, 1:] - sxx[k0:, 1:, :-1]) / c.dx, 0, 0, w)
        d = d + self.pml("sxy", (sxy[k0:, 1:, 1:] - sxy[k0:, :-1, 1:]) / c.dy, 1, 0, w)
        d = d + self.pml("sxz", (sxz[k0:] - below)[:, 1:, 1:] / c.dz, 2, 0, w)
        vx[w] += dt / ((rho[w] + rho[k0:, 1:, :-1]) / 2) * d
        w = (slice(k0, nz), slice(0, ny - 1), slice(0, nx - 1))
        below = torch.cat([-syz[:1], syz[:-1]])[k0:]
        d = self.pml("syx", (sxy[k0:, :-1, 1:] - sxy[k0:, :-1, :-1]) / c.dx, 0, 1, w)
        d = d + self.pml("syy", (syy[k0:, 1:, :-1] - syy[k0:, :-1, :-1]) / c.dy, 1, 1, w)
        d = d + self.pml("syz", (syz[k0:] - below)[:, :-1, :-1] / c.dz, 2, 0, w)
        vy[w] += dt / ((rho[w] + rho[k0:, 1:, :-1]) / 2) * d
        w = (slice(0, nz - 1), slice(1, ny), slice(0, nx - 1))
        d = self.pml("szx", (sxz[:-1, 1:, 1:] - sxz[:-1, 1:, :-1]) / c.dx, 0, 1, w)
        d = d + self.pml("szy", (syz[:-1, 1:, :-1] - syz[:-1, :-1, :-1]) / c.dy, 1, 0, w)
        d = d + self.pml("szz", (szz[1:, 1:, :-1] - szz[:-1, 1:, :-1]) / c.dz, 2, 1, w)
        vz[w] += dt / ((rho[w] + rho[1:, 1:, :-1]) / 2) * d
        if c.dirichlet:
            for v in (vx, vy, vz):
                v[:, 0] = v[:, -1] = v[-1] = 0
                v[:, :, 0] = v[:, :, -1] = 0
                if not c.free_surface:
                    v[0] = 0

    def energy(self):
        c, p = self.c, self.c.npoints_pml
        b = (slice(p, c.nz - 1 - p), slice(p, c.ny - 1 - p), slice(p, c.nx - 1 - p))
        rho, cp, cs = self.rho[b], self.cp[b], self.cs[b]
        vx, vy, vz, sxx, syy, szz, sxy, sxz, syz = (f[b] for f in self.f)
        mu, lam = rho * cs * cs, rho * (cp * cp - 2.0 * cs * cs)
        ss = sxx * sxx + syy * syy + szz * szz + 2.0 * (sxy * sxy + sxz * sxz + syz * syz)
        tr = sxx + syy + szz
        pot = 0.5 * (ss / (2.0 * mu) - lam * tr * tr / (2.0 * mu * (3.0 * lam + 2.0 * mu)))
        vol = c.dx * c.dy * c.dz
        return [float((0.5 * rho * (vx * vx + vy * vy + vz * vz)).sum()) * vol, float(pot.sum()) * vol]

    def source(self, it):
        c, (k, j, i) = self.c, (self.c.ksrc, self.c.jsrc, self.c.isrc)
        a, u = math.pi ** 2 * c.f0 ** 2, (it - 1) * c.dt - c.t0_effective
        g = c.factor * math.exp(-a * u * u)
        s = {ela.WAVELET_GAUSSIAN: g, ela.WAVELET_DGAUSSIAN: -2.0 * a * u * g}.get(c.wavelet, (1.0 - 2.0 * a * u * u) * g)
        th = math.radians(c.angle_force)
        fx, fy = math.sin(th) * s, math.cos(th) * s
        rho, f = self.rho, self.f
        if c.src_kind in (ela.SRC_FORCE, ela.SRC_FORCE3):
            amp = (fx, fy, 0.0) if c.src_kind == ela.SRC_FORCE else (s, s, s)
            for q, (v, o) in enumerate(zip(amp, ((k, j, i - 1), (k, j + 1, i), (k + 1, j, i)))):
                f[q][k, j, i] += v * c.dt / ((rho[k, j, i] + rho[o]) / 2)
        else:
            amp = (fx, fx, fy) if c.src_kind == ela.SRC_REFERENCE_SIGMA else (s, s, s)
            for q, v in zip((3, 4, 5), amp):
                f[q][k, j, i] += v * c.dt * rho[k, j, i] * self.cp[k, j, i] ** 2

    def run(self, n):
        """n steps from rest: (seismograms [nstep / sample_every][nrec][3], energy)."""
        c = self.c
        i, j, k = torch.as_tensor(np.asarray(c.receivers).T.astype(np.int64), device=self.dev)
        seis = torch.zeros(c.nstep // c.sample_every, c.nrec, 3, dtype=torch.float64, device=self.dev)
        en = np.zeros((c.nstep // c.energy_every if c.energy_every else 0, 2))
        for it in range(1, n + 1):
            self.stress()
            self.velocity()
            if it % c.sample_every == 0 and it // c.sample_every <= len(seis):
                seis[it // c.sample_every - 1] = torch.stack([v[k, j, i] for v in self.f[:3]], 1)
            if c.energy_every and it % c.energy_every == 0 and it // c.energy_every <= len(en):
                en[it // c.energy_every - 1] = self.energy()
            if it <= c.nstep:
                self.source(it)
        return seis.cpu().numpy(), en


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "serve":
        return [_Plain(cfg, model, dev).run(cfg.nstep)[0] for cfg, model in _serve_shots(case, seed)]
    p = _Plain(*_shot(case, seed), dev)
    seis, en = p.run(case["warm"] + case["steps"])
    return {"vz": p.f[2].cpu().numpy()} if case["kind"] == "look" else {"seismograms": seis, "energy": en}
