"""The work of a user of this framework whose speed is measured, case by case.

A user's program is a time loop: it makes a ``Solver``, uploads a state, and calls
``step`` (three Runge-Kutta substeps) thousands of times, reading the state back
every few hundred steps.  So most cases are one such step on a state that stays
on the device, from grids whose kernels last microseconds (``dns_32``) to the
largest LES of the benchmark (512x257x512).  The other two are the transform
entry point for callers with device arrays, and one epoch of the learned
closure's training.

Sizes: the transforms take powers of two in x and z (16 to 512 here), the
wall-normal direction any number of rows, so that is where the odd sizes are.
"""
import math

import numpy as np
import torch

from diablo3_amd import closure, configs, ic
from diablo3_amd.config import FP64, MIXED
from diablo3_amd.problem import Problem
from diablo3_amd.solver import Solver, load


def _step(name, flow, nx, ny, nz, precision, scalars=1):
    return {"name": name, "kind": "step", "flow": flow, "nx": nx, "ny": ny, "nz": nz, "scalars": scalars,
            "precision": precision}


def listed():
    return [
        # the grid of the quick checks: every kernel is shorter than its launch
        _step("dns_32_fp64", "dns", 32, 33, 32, "fp64"),
        # the small front of the first DNS configuration; latency still counts
        _step("dns_64_fp64", "dns", 64, 65, 64, "fp64"),
        # an elongated domain with two scalars and a row count that no tile divides
        _step("dns_128x97x64_mixed_2th", "dns", 128, 97, 64, "mixed", 2),
        # the flagship DNS, in both precisions
        _step("dns_256_fp64", "dns", 256, 129, 256, "fp64"),
        _step("dns_256_mixed", "dns", 256, 129, 256, "mixed"),
        # the coarse LES that follows a filtered DNS
        _step("les_128_fp64", "les", 128, 129, 128, "fp64"),
        # the three runs that the benchmark compares: FP64 with the AMD closure, mixed
        # with it, mixed with the learned closure
        _step("les_512_fp64", "les", 512, 257, 512, "fp64"),
        _step("les_512_mixed", "les", 512, 257, 512, "mixed"),
        _step("les_512_mixed_learned", "learned", 512, 257, 512, "mixed"),
        # one field to Fourier space in the caller's own device memory
        {"name": "to_fourier_128x97x128", "kind": "transform", "nx": 128, "ny": 97, "nz": 128},
        # one epoch of the closure's training on a snapshot's worth of samples
        {"name": "train_epoch_1m", "kind": "train", "samples": 1040385, "batch": 16384},
    ]


def draw(rng):
    kind = rng.choices(["dns", "les", "learned", "transform", "train"], [5, 3, 1, 1, 1])[0]
    if kind == "train":
        return {"kind": "train", "samples": int(math.exp(rng.uniform(math.log(3e4), math.log(2e6)))),
                "batch": rng.choice([1024, 4096, 16384])}
    if kind == "transform":
        nx, nz = rng.choice([32, 64, 128]), rng.choice([32, 64, 128])
        return {"kind": "transform", "nx": nx, "ny": rng.randrange(17, 130), "nz": nz}
    nx, nz = rng.choice([32, 64, 128, 256, 512]), rng.choice([32, 64, 128, 256])
    ny = int(round(math.exp(rng.uniform(math.log(17), math.log(257)))))
    precision = rng.choice(["fp64", "mixed"])
    scalars = 1
    if kind == "dns":
        # 512 points in x with two scalars exceed the FP64 x pass and are refused
        scalars = rng.choice([0, 1, 1, 2] if nx < 512 or precision == "mixed" else [0, 1, 1])
    c = _step("", kind, nx, ny, nz, precision, scalars)
    del c["name"]
    return c


# ---------------------------------------------------------------------------------
# a user's program
# ---------------------------------------------------------------------------------
def _config(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    large = nx >= 256
    precision = MIXED if case.get("precision") == "mixed" else FP64
    if case.get("flow", "dns") == "dns":
        c = configs.front_dns(nx, ny, nz, 2000.0 if large else 1000.0, 0.5, 0.25 if large else 1.0, 1.0,
                              5e-4 if large else 1e-3, 1e-3, precision)
        n = case.get("scalars", 1)
        if n != 1:
            c = c.copy(n_th=n, ri=c.ri * n, pr=[1.0, 0.7][:n], create_new_th=[True] * n,
                       th_bc_ymin=c.th_bc_ymin * n, th_bc_ymin_c1=c.th_bc_ymin_c1 * n,
                       th_bc_ymax=c.th_bc_ymax * n, th_bc_ymax_c1=c.th_bc_ymax_c1 * n,
                       dthdx=c.dthdx * n, dthdz=[0.0] * n).derive()
        return c
    c = configs.front_les(nx, ny, nz, 1e5 if large else 5000.0, 2e-4, 1e-2, precision=precision)
    return c.copy(les_model_type=6) if case["flow"] == "learned" else c


def _spectrum(cfg, phys):
    """The kept modes of a physical field [j][z][x]."""
    h = torch.fft.rfft(phys, dim=2)[:, :, :cfg.kxr] / cfg.nx
    f = torch.fft.fft(h, dim=1) / cfg.nz
    return torch.cat([f[:, :cfg.nkz + 1], f[:, cfg.nz - cfg.nkz:]], dim=1)


def _initial(p, seed):
    """The configuration's front with seeded noise in the velocity and the scalars,
    before the projection (compact Fourier arrays on the host)."""
    cfg = p.cfg
    gen = torch.Generator("cuda").manual_seed(seed)
    shape = (cfg.ny2, cfg.nz, cfg.nx)

    def noise(amplitude):
        return (torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64) - 0.5) * amplitude

    y = torch.as_tensor(p.met["gyf"], device="cuda") - 0.5 * cfg.ly
    x = torch.arange(cfg.nx, device="cuda", dtype=torch.float64) * (cfg.lx / cfg.nx) - 0.5 * cfg.lx
    u3 = torch.zeros((cfg.ny2, 1, cfg.nx), device="cuda", dtype=torch.float64)
    ths = []
    rows = torch.zeros((cfg.ny2, 1, 1), device="cuda", dtype=torch.float64)
    rows[1:cfg.ny + 1] = 1.0
    for n in range(cfg.n_th):
        if cfg.ic_type == 4:  # uniform stratification
            ths.append((cfg.ri[n] * y)[:, None, None].expand(-1, 1, cfg.nx))
        else:  # a front in thermal-wind balance
            s = math.hypot(cfg.ri[n], cfg.ro_inv)
            t = torch.tanh((x[None] * cfg.ro_inv + y[:, None] * cfg.ri[n]) / (cfg.delta * s))
            ths.append((s * t - 2.0 * cfg.ro_inv / cfg.lx * x[None])[:, None, :])
            u3 = (cfg.delta * s / cfg.ri[n] * t - 2.0 * cfg.delta / cfg.lx * y[:, None])[:, None, :]
    spec = [_spectrum(cfg, b + noise(cfg.kick)).cpu().numpy() for b in (0.0 * u3, 0.0 * u3, u3)]
    cth = [_spectrum(cfg, (t + noise(2e-3)) * rows).cpu().numpy() for t in ths]
    s = ic.FourierState(*spec, np.zeros_like(spec[0]), cth)
    ic.apply_bc_vel_post(cfg, p.met, s)
    return s


def _samples(case, seed):
    """Features and targets of the closure's training: 13 live features, a target
    that depends on them, and noise."""
    gen = torch.Generator("cuda").manual_seed(seed)
    n = case["samples"]
    x = torch.zeros((n, 16), device="cuda")
    x[:, :13] = torch.randn((n, 13), generator=gen, device="cuda")
    t = torch.stack([torch.tanh(x[:, 0] + 0.5 * x[:, 3]), 0.3 * x[:, 1] * x[:, 5]], dim=1)
    t = t + 0.1 * torch.randn((n, 2), generator=gen, device="cuda")
    return x.cpu().numpy(), t.cpu().numpy()


class _Fields(list):
    """The fields of a solver's state: u1, u2, u3, p and the scalars.  The state is
    the handle's own device memory, which a time loop does not read back after a
    step; it is read (``download_state``) when somebody looks at the fields, in the
    precision in which the handle carries its fields through physical space."""

    def __init__(self, solver):
        super().__init__()
        self.solver = solver

    def __len__(self):
        return 4 + self.solver.cfg.n_th

    def __getitem__(self, k):
        return list(self)[k]

    def __iter__(self):
        s = self.solver.download_state()
        as_held = np.complex64 if self.solver.cfg.precision == MIXED else np.complex128
        return iter([a.astype(as_held) for a in (s.cu1, s.cu2, s.cu3, s.cp, *s.cth)])


def prepare(case, seed):
    if case["kind"] == "train":
        m = closure.Mlp(seed=7)
        x, t = _samples(case, seed)
        m.set_norm(closure.make_norm(x[:200000]))
        m.set_data(x, t)
        return {"kind": "train", "mlp": m, "batch": case["batch"], "epoch": 0}
    cfg = _config(case)
    p = Problem(cfg)
    g = Solver(p)
    if case["kind"] == "transform":
        gen = torch.Generator("cuda").manual_seed(seed)
        phys = torch.randn((cfg.ny2, cfg.nz + 2, cfg.nx + 2), generator=gen, device="cuda", dtype=torch.float64)
        four = torch.zeros((cfg.ny2, cfg.nz + 2, cfg.nxp + 1), device="cuda", dtype=torch.complex128)
        torch.cuda.synchronize()
        return {"kind": "transform", "solver": g, "phys": phys, "four": four}
    if case["flow"] == "learned":
        params, norm, _ = closure.load_params()
        g.set_closure(params, norm)
    g.upload_state(_initial(p, seed))
    g.rem_div()
    torch.cuda.empty_cache()
    return {"kind": "step", "solver": g, "n": 0, "time": 0.0}


def run(state):
    if state["kind"] == "train":
        m = state["mlp"]
        loss = m.train(1, state["batch"], lr=1e-3, seed=state["epoch"])
        state["epoch"] += 1
        return {"params": m.params, "loss": loss}
    g = state["solver"]
    if state["kind"] == "transform":
        rc = load().dgpu_fft_xz_to_fourier_noalloc(g.h, state["phys"].data_ptr(), state["four"].data_ptr())
        if rc:
            raise RuntimeError(load().dgpu_last_error().decode())
        return state["four"][:, :g.cfg.kzr]
    state["n"] += 1
    # LES: as a restarted run, so that the closure is on from the first step
    g.step(time=state["time"], time_step=state["n"], create_new_flow=not g.cfg.use_les)
    state["time"] += g.cfg.delta_t
    return _Fields(g)


def work(case):
    if case["kind"] == "train":
        n = case["samples"]
        macs = 13 * 64 + 64 * 64 + 64 * 2
        return {"bytes": n * (16 + 2) * 4, "flops": 3 * 2 * macs * n}
    cfg = _config(case)
    points = cfg.nx * cfg.nz * cfg.ny2
    mode = cfg.kxr * cfg.kzr * cfg.ny2 * 16

    def transform():  # one real two-dimensional transform of every plane
        return 2.5 * points * math.log2(cfg.nx * cfg.nz)

    if case["kind"] == "transform":
        return {"bytes": 8 * points + (cfg.nxp + 1) * cfg.kzr * cfg.ny2 * 16, "flops": transform()}
    # each substep depends on all of the one before: it reads the state and leaves
    # the next one; the Runge-Kutta memory is written by substeps 1 and 2 and read
    # by 2 and 3
    nf = 3 + cfg.n_th
    transforms = nf + 8 + 3 * cfg.n_th
    if cfg.use_les:
        transforms += 4 * nf
    if case["flow"] == "learned":
        extra = 2 * (13 * 64 + 64 * 64 + 64 * 2) * points
    else:
        extra = 0
    return {"bytes": 3 * 2 * (nf + 1) * mode + 4 * nf * mode, "flops": 3 * (transforms * transform() + extra)}


# ---------------------------------------------------------------------------------
# the same in 64 bits with torch alone
# ---------------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "train":
        return None  # the network's BF16 operands are part of its definition
    if case["kind"] == "transform":
        cfg = _config(case)
        gen = torch.Generator("cuda").manual_seed(seed)
        phys = torch.randn((cfg.ny2, cfg.nz + 2, cfg.nx + 2), generator=gen, device="cuda", dtype=torch.float64)
        out = torch.zeros((cfg.ny2, cfg.kzr, cfg.nxp + 1), device="cuda", dtype=torch.complex128)
        out[:, :, :cfg.kxr] = _spectrum(cfg, phys[:, :cfg.nz, :cfg.nx])
        return out
    if case["flow"] == "learned":
        return None  # BF16 network behind an envelope that a last bit can cross
    p = Problem(_config(case))
    e = _Exact(p, _initial(p, seed))
    e.project(None)
    for rk in (1, 2, 3):
        e.substep(rk)
    return [a.cpu().numpy() for a in (e.u[0], e.u[1], e.u[2], e.p, *e.u[3:])]


class _Exact:
    """One RKW3 / Crank-Nicolson step of the staggered channel, field by field, the
    wall-normal index first: u1, u3 and the scalars at GYF, u2 at GY."""

    def __init__(self, p, s):
        self.c = p.cfg

        def dev(a):
            return torch.as_tensor(np.asarray(a), device="cuda")

        self.kx = dev(p.kx[:self.c.kxr])[None, None, :]
        self.kz = dev(p.kz)[None, :, None]
        self.gy, self.gyf, self.dy, self.dyf = (dev(p.met[k])[:, None, None] for k in ("gy", "gyf", "dy", "dyf"))
        self.u = [dev(a).clone() for a in (s.cu1, s.cu2, s.cu3, *s.cth)]
        self.p = dev(s.cp).clone()
        self.cf = [torch.zeros_like(self.p) for _ in self.u]

    # ---- transforms of all planes
    def phys(self, f):
        c = self.c
        z = torch.zeros((f.shape[0], c.nz, c.kxr), dtype=torch.complex128, device="cuda")
        z[:, :c.nkz + 1] = f[:, :c.nkz + 1]
        z[:, c.nz - c.nkz:] = f[:, c.nkz + 1:]
        h = torch.fft.ifft(z, dim=1) * c.nz
        h[:, :, 0] = h[:, :, 0].real + 0j
        return torch.fft.irfft(h, n=c.nx, dim=2) * c.nx

    def four(self, r):
        return _spectrum(self.c, r)

    # ---- one substep
    def substep(self, rk):
        c, ny = self.c, self.c.ny
        h = c.delta_t * (8.0, 2.0, 5.0)[rk - 1] / 15.0
        beta, zeta = (1.0, 25.0 / 8.0, 9.0 / 4.0)[rk - 1], (0.0, -17.0 / 8.0, -5.0 / 4.0)[rk - 1]
        sgs = None
        if c.use_les:
            self.wall_rows()
            sgs = self.amd()
        nl = self.nonlinear(sgs)
        rhs = []
        for e in range(len(self.u)):
            cf = self.explicit(e) + nl[e]
            r = self.u[e] + beta * h * cf + zeta * h * self.cf[e] - h * self.gradient(e)
            r = r + 0.5 * h * self.diffusivity(e) * c.nu_v_scale * self.d2(e, self.u[e])
            lo, hi = self.rows(e)
            r[:lo] = 0
            r[hi + 1:] = 0
            rhs.append(r)
            self.cf[e][lo:hi + 1] = cf[lo:hi + 1]
        del nl
        for e in [*range(3, len(self.u)), 1, 0, 2]:
            visc = None if sgs is None else sgs["nu"] if e < 3 else sgs["kappa"][e - 3]
            self.crank_nicolson(e, rhs[e], h, visc)
        self.project(h)

    def rows(self, e):
        c = self.c
        if e == 1:
            return 2, c.ny
        return (c.jstart, c.ny) if e < 3 else (c.jstart_th[e - 3], c.ny)

    def diffusivity(self, e):
        return self.c.nu if e < 3 else self.c.nu / self.c.pr[e - 3]

    def d2(self, e, f):
        out = torch.zeros_like(f)
        dy, dyf = self.dy, self.dyf
        if e == 1:
            out[2:-1] = ((f[3:] - f[2:-1]) / dyf[2:-1] - (f[2:-1] - f[1:-2]) / dyf[1:-2]) / dy[2:-1]
        else:
            out[1:-1] = ((f[2:] - f[1:-1]) / dy[2:] - (f[1:-1] - f[:-2]) / dy[1:-1]) / dyf[1:-1]
        return out

    def gradient(self, e):
        if e >= 3:
            return 0.0
        if e == 0:
            return 1j * self.kx * self.p
        if e == 2:
            return 1j * self.kz * self.p
        out = torch.zeros_like(self.p)
        out[1:] = (self.p[1:] - self.p[:-1]) / self.dy[1:]
        return out

    def explicit(self, e):
        c, u = self.c, self.u
        f = u[e]
        k2 = (self.kx ** 2 + self.kz ** 2) ** c.beta
        cf = -self.diffusivity(e) * k2 * f
        wind = c.flavor == "Front" and c.ro_inv != 0.0
        cori = c.ro_inv / c.delta
        if e in (0, 2):
            cf = cf + (cori * u[2] if e == 0 else -cori * u[0])
            for n in range(c.n_th):
                cf = cf + (c.grav_x if e == 0 else c.grav_z) * u[3 + n]
        elif e == 1:
            for n in range(c.n_th):
                t = u[3 + n]
                b = torch.zeros_like(f)
                b[1:] = (t[1:] * self.dyf[:-1] + t[:-1] * self.dyf[1:]) / (2.0 * self.dy[1:])
                b[:, 0, 0] = 0
                cf = cf + c.grav_y * b
        else:
            cf = cf - c.dthdx[e - 3] * u[0] - c.dthdz[e - 3] * u[2]
        if wind:
            u2c = torch.zeros_like(f)
            u2c[:-1] = 0.5 * (u[1][:-1] + u[1][1:])
            y = (self.gy if e == 1 else self.gyf) - 0.5 * c.ly
            for n in [e - 3] if e >= 3 else range(c.n_th):
                sx, sz = c.dthdx[n] * c.delta / c.ro_inv, -c.dthdz[n] * c.delta / c.ro_inv
                cf = cf - sx * y * 1j * self.kz * f - sz * y * 1j * self.kx * f
                if e == 0:
                    cf = cf - sz * u2c
                elif e == 2:
                    cf = cf - sx * u2c
        return cf

    def nonlinear(self, sgs):
        c, ny, dy, dyf = self.c, self.c.ny, self.dy, self.dyf
        v = [self.phys(f) for f in self.u]
        out = []
        for e in range(len(v)):
            f = v[e]
            nl = torch.zeros_like(self.p)
            lo, hi = self.rows(e)
            a, up, dn = slice(lo, hi + 1), slice(lo + 1, hi + 2), slice(lo - 1, hi)
            if e == 1:
                u1 = (dyf[a] * v[0][a] + dyf[dn] * v[0][dn]) / (2.0 * dy[a])
                u3 = (dyf[a] * v[2][a] + dyf[dn] * v[2][dn]) / (2.0 * dy[a])
                px, pz = u1 * f[a], u3 * f[a]
                flux = (0.25 * (f[a] + f[up]) ** 2 - 0.25 * (f[a] + f[dn]) ** 2) / dy[a]
            else:
                px, pz = f[a] * v[0][a], f[a] * v[2][a]
                flux = 0.5 * ((f[up] + f[a]) * v[1][up] - (f[a] + f[dn]) * v[1][a]) / dyf[a]
            if sgs is not None:
                ax, az, ay = sgs["add"][e]
                px, pz = px + ax[a], pz + az[a]
                flux = flux if ay is None else flux + ay[a]
            nl[a] = -1j * self.kx * self.four(px) - 1j * self.kz * self.four(pz) - self.four(flux)
            out.append(nl)
        return out

    # ---- Crank-Nicolson: rows 0..ny+1, the wall rows as boundary conditions
    def crank_nicolson(self, e, rhs, h, visc):
        c, ny = self.c, self.c.ny
        n2 = ny + 2
        t, t2 = 0.5 * h * self.diffusivity(e) * c.nu_v_scale, 0.5 * h
        lo, hi = self.rows(e)
        names = "uvw"[e] if e < 3 else None
        if names:
            kind = [getattr(c, names + "_bc_" + w) for w in ("ymin", "ymax")]
            val = [getattr(c, names + "_bc_" + w + "_c1") for w in ("ymin", "ymax")]
        else:
            kind = [c.th_bc_ymin[e - 3], c.th_bc_ymax[e - 3]]
            val = [c.th_bc_ymin_c1[e - 3], c.th_bc_ymax_c1[e - 3]]
        # boundary rows: row -> (lower, diagonal, upper, value)
        bc = {}
        if e == 1:
            bc[0] = (0.0, 1.0, 0.0, 0.0)
            for j in (1, 2):
                bc[j] = (0.0, 1.0, 0.0, val[0])
            for j in (ny, ny + 1):
                bc[j] = (0.0, 1.0, 0.0, val[1])
        else:
            bc[0] = bc[ny + 1] = (0.0, 1.0, 0.0, 0.0)
            bc[1] = (0.0, 1.0, 0.0, val[0]) if kind[0] == 0 else (0.0, -1.0, 1.0, float(self.dy[2]) * val[0])
            bc[ny] = (0.0, 1.0, 0.0, val[1]) if kind[1] == 0 else (-1.0, 1.0, 0.0, float(self.dy[ny]) * val[1])
        dy, dyf = [x.flatten().tolist() for x in (self.dy, self.dyf)]

        def faces(j):
            if e == 1:
                return 1.0 / (dyf[j - 1] * dy[j]), 1.0 / (dyf[j] * dy[j])
            return 1.0 / (dy[j] * dyf[j]), 1.0 / (dy[j + 1] * dyf[j])

        wlo, whi = lo - 1, hi + 1
        if visc is None:  # the same matrix for every mode
            m = torch.zeros((n2, n2), dtype=torch.complex128, device="cuda")
            for j in range(n2):
                if j in bc:
                    l, d, up, value = bc[j]
                    rhs[j] = 0
                    rhs[j, 0, 0] = value
                elif lo <= j <= hi:
                    il, iu = faces(j)
                    l, d, up = -t * il, 1.0 + t * (il + iu), -t * iu
                else:
                    l, d, up = 0.0, 1.0, 0.0
                m[j, j] = d
                if j > 0:
                    m[j, j - 1] = l
                if j < ny + 1:
                    m[j, j + 1] = up
            x = torch.linalg.solve(m, rhs.reshape(n2, -1)).reshape(rhs.shape)
            self.u[e][wlo:whi + 1] = x[wlo:whi + 1]
            return
        # an eddy viscosity: one system for every physical column
        r, f = self.phys(rhs), self.phys(self.u[e])
        x = torch.empty_like(r)
        ups, piv = [None] * n2, [None] * n2
        for j in range(n2):
            if j in bc:
                l, d, up, b = bc[j]
                d = torch.full_like(r[j], d)
                b = torch.full_like(r[j], b)
            elif lo <= j <= hi:
                il, iu = faces(j)
                nl_ = 0.5 * (visc[j] + visc[j - 1]) if e == 1 else visc[j]
                nu_ = 0.5 * (visc[j] + visc[j + 1]) if e == 1 else (visc[j + 1])
                low, high = (t + t2 * nl_) * il, (t + t2 * nu_) * iu
                l, d, up = -low, 1.0 + low + high, -high
                b = r[j] + t2 * (nu_ * (f[j + 1] - f[j]) * iu - nl_ * (f[j] - f[j - 1]) * il)
            else:
                l, d, up, b = 0.0, torch.ones_like(r[j]), 0.0, torch.zeros_like(r[j])
            if j > 0:
                q = -l / piv[j - 1]
                d = d + q * ups[j - 1]
                b = b + q * x[j - 1]
            piv[j], ups[j] = d, up
            x[j] = b
        x[ny + 1] = x[ny + 1] / piv[ny + 1]
        for j in range(ny, -1, -1):
            x[j] = (x[j] - ups[j] * x[j + 1]) / piv[j]
        f[wlo:whi + 1] = x[wlo:whi + 1]
        self.u[e] = self.four(f)

    # ---- projection (and, with the substep's length h, the pressure update)
    def project(self, h):
        c, ny, dy, dyf = self.c, self.c.ny, self.dy, self.dyf
        ikx, ikz = 1j * self.kx, 1j * self.kz
        k2 = (self.kx ** 2 + self.kz ** 2)[0]
        d = ikx * self.u[0] + ikz * self.u[2]
        d[1:-1] = d[1:-1] + (self.u[1][2:] - self.u[1][1:-1]) / dyf[1:-1]
        phi = torch.zeros_like(self.p)
        piv, ups = [None] * (ny + 1), [None] * (ny + 1)
        zero = torch.zeros_like(k2)
        for j in range(1, ny + 1):
            if j == 1:
                a, b, up, r = zero, zero - 1.0, zero + 1.0, torch.zeros_like(phi[0])
                b[0, 0], up[0, 0] = 1.0, 0.0
            elif j == ny:
                a, b, up, r = zero + 1.0, zero - 1.0, zero, torch.zeros_like(phi[0])
            else:
                lo, hi = 1.0 / (dy[j] * dyf[j]), 1.0 / (dy[j + 1] * dyf[j])
                a, b, up, r = zero + lo, -(lo + hi) - k2, zero + hi, d[j]
            if j > 1:
                q = -a / piv[j - 1]
                b = b + q * ups[j - 1]
                r = r + q * phi[j - 1]
            piv[j], ups[j] = b, up
            phi[j] = r
        phi[ny] = phi[ny] / piv[ny]
        for j in range(ny - 1, 0, -1):
            phi[j] = (phi[j] - ups[j] * phi[j + 1]) / piv[j]
        i = slice(1, ny + 1)
        self.u[0][i] -= ikx * phi[i]
        self.u[2][i] -= ikz * phi[i]
        self.u[1][2:ny + 1] -= (phi[2:ny + 1] - phi[1:ny]) / dy[2:ny + 1]
        if h is not None:
            self.p[c.jstart:ny + 1] += phi[c.jstart:ny + 1] / h

    # ---- LES: the wall and ghost rows of the state, then the AMD closure
    def wall_rows(self):
        c, ny, u = self.c, self.c.ny, self.u
        for e in (0, 2, *range(3, len(u))):
            f = u[e]
            if e < 3:
                name = "uvw"[e]
                klo, khi = getattr(c, name + "_bc_ymin"), getattr(c, name + "_bc_ymax")
                vlo, vhi = getattr(c, name + "_bc_ymin_c1"), getattr(c, name + "_bc_ymax_c1")
            else:
                klo, khi, vlo, vhi = (getattr(c, k)[e - 3] for k in ("th_bc_ymin", "th_bc_ymax", "th_bc_ymin_c1",
                                                                    "th_bc_ymax_c1"))
            if klo == 0:
                f[0:2] = 0
                f[0:2, 0, 0] = vlo
            else:  # with the closure on, the ghost rows copy the first interior one
                f[1] = f[2]
                f[0] = f[2]
            if khi == 0:
                f[ny:] = 0
                f[ny:, 0, 0] = vhi
                if e == 2:
                    f[ny + 1, 0, 0] = 0
            else:
                f[ny] = f[ny - 1]
                f[ny + 1] = f[ny - 1]
        # u2 is Dirichlet at both walls of these flows
        u[1][1] = 2.0 * c.v_bc_ymin_c1 - u[1][2]
        u[1][0] = u[1][1]
        u[1][ny + 1, 0, 0] = 2.0 * c.v_bc_ymax_c1 - u[1][ny, 0, 0]

    def amd(self):
        c, ny, dy, dyf = self.c, self.c.ny, self.dy, self.dyf
        v = [self.phys(f) for f in self.u]
        vx = [self.phys(1j * self.kx * f) for f in self.u]
        vz = [self.phys(1j * self.kz * f) for f in self.u]
        ax, az = 3.0 * c.lx / c.nx, 3.0 * c.lz / c.nz
        ay = 2.0 * dy.clone()
        ay[0] = 1.0
        ayf = 2.0 * dyf

        def width(w):
            return -2.0 * 0.2887 ** 2 * 3.0 / (1.0 / ax ** 2 + 1.0 / w ** 2 + 1.0 / az ** 2)

        def up(f):  # difference of a GYF field, at GY
            o = torch.zeros_like(f)
            o[1:] = (f[1:] - f[:-1]) / dy[1:]
            return o

        def at_gyf(f):  # mean of the two GY neighbours
            o = torch.zeros_like(f)
            o[:-1] = 0.5 * (f[:-1] + f[1:])
            return o

        def at_gy(f):  # interpolation of a GYF field
            o = torch.zeros_like(f)
            o[1:] = (f[1:] * dyf[:-1] + f[:-1] * dyf[1:]) / (2.0 * dy[1:])
            return o

        d2 = torch.zeros_like(v[1])
        d2[:-1] = (v[1][1:] - v[1][:-1]) / dyf[:-1]
        d1y, d3y = up(v[0]), up(v[2])

        def coefficient(f):
            """max(0, -G_ik G_jk S_ij) / |G|^2 of the scaled gradient G."""
            a1, a2, a3, a4, a5, a6, o4, o5, o6 = f
            s = torch.stack([a1, a4, a5, a4, a2, a6, a5, a6, a3]).reshape(3, 3, *a1.shape)
            z = torch.zeros_like(a1)
            o = torch.stack([z, o4, o5, -o4, z, o6, -o5, -o6, z]).reshape(3, 3, *a1.shape)
            # tr S^3 + tr(S O O^T) of the symmetric part
            t = sum(s[i, k] * (s[i, l] * s[l, k] + o[i, l] * o[k, l]) for i in range(3) for k in range(3)
                    for l in range(3))
            n = (s * s).sum((0, 1)) + (o * o).sum((0, 1))
            return torch.where(t < 0, -t / torch.where(n > 0, n, 1.0), 0.0)

        # entries at GYF: 11, 22, 33, 13; at GY: 12, 23 (first index scaled)
        g = [vx[0], d2, vz[2], 0.5 * (vz[0] * (az / ax) + vx[2] * (ax / az)),
             0.5 * (vz[0] * (az / ax) - vx[2] * (ax / az))]
        k = [0.5 * (d1y * (ay / ax) + vx[1] * (ax / ay)), 0.5 * (vz[1] * (az / ay) + d3y * (ay / az)),
             0.5 * (d1y * (ay / ax) - vx[1] * (ax / ay)), 0.5 * (vz[1] * (az / ay) - d3y * (ay / az))]

        def by_rows(make):
            """coefficient() on slabs of rows, to bound the memory."""
            out = torch.zeros_like(v[0])
            for j in range(0, ny + 2, 16):
                out[j:j + 16] = coefficient([f[j:j + 16] for f in make])
            return out

        i = [at_gy(f) for f in g]
        c_gy = by_rows([i[0], i[1], i[2], k[0], i[3], k[1], k[2], i[4], k[3]])
        m = [at_gyf(f) for f in k]
        c_gyf = by_rows([g[0], g[1], g[2], m[0], g[3], m[1], m[2], g[4], m[3]])
        del i, m, g, k
        w_gy, w_gyf = width(ay), width(ayf)
        js = c.jstart
        inner = torch.zeros_like(dy)
        inner[3:ny] = 1.0
        nu = -0.5 * w_gy * c_gy * inner

        def stress(dudy, du2):  # the stress at GY (row 1 keeps its strain)
            t = w_gy * c_gy * 0.5 * du2
            t[1] = w_gy[1] * 0.5 * (dudy[1] + du2[1])
            return t

        t12, t23 = stress(d1y, vx[1]), stress(d3y, vz[1])
        rows_f = torch.zeros_like(dy)
        rows_f[js:ny] = 1.0
        rows_g = torch.zeros_like(dy)
        rows_g[2:ny + 1] = 1.0
        cw = w_gyf * c_gyf * rows_f

        def dflux(t):
            o = torch.zeros_like(t)
            o[:-1] = (t[1:] - t[:-1]) / dyf[:-1]
            return o * rows_f

        t13 = cw * 0.5 * (vz[0] + vx[2])
        add = [(cw * vx[0], t13, dflux(t12)), ((t12 - nu * d1y) * rows_g, (t23 - nu * d3y) * rows_g, None),
               (t13, cw * vz[2], dflux(t23))]
        kappa = []
        for n in range(c.n_th):
            t, tx, tz = v[3 + n], vx[3 + n], vz[3 + n]
            ty = up(t)

            def scalar(y, dx1, dy1, dz1, dx2, dy2, dz2, dx3, dy3, dz3, bx, by, bz):
                """max(0, -(delta_k du_i/dx_k)(delta_k dth/dx_k) dth/dx_i) / |delta dth|^2."""
                w = [ax, y, az]
                grad = [[dx1, dy1, dz1], [dx2, dy2, dz2], [dx3, dy3, dz3]]
                b = [bx, by, bz]
                q = -sum(w[m] ** 2 * grad[l][m] * b[m] * b[l] for l in range(3) for m in range(3))
                nrm = sum((w[m] * b[m]) ** 2 for m in range(3))
                return torch.where(q > 0, q / torch.where(nrm > 0, nrm, 1.0), 0.0)

            at = at_gy
            cg = scalar(ay, at(vx[0]), d1y, at(vz[0]), vx[1], at(d2), vz[1], at(vx[2]), d3y, at(vz[2]), at(tx), ty,
                        at(tz))
            kappa.append(-0.5 * w_gy * cg * inner)
            at = at_gyf
            cg = scalar(ayf, vx[0], at(d1y), vz[0], at(vx[1]), d2, at(vz[1]), vx[2], at(d3y), vz[2], tx, at(ty), tz)
            row = torch.zeros_like(dy)
            row[c.jstart_th[n]:ny + 1] = 1.0
            f = 0.5 * w_gyf * cg * row
            add.append((f * tx, f * tz, None))
        return {"nu": nu, "kappa": kappa, "add": add}
