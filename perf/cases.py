"""The work a user of this framework has it do, as cases to time.

Every case goes through the package's Solver (or, for the field reads, the C
entry point fen_download into host arrays that the program keeps, as the
Fortran modules do with their host mirrors).  A run case is a stretch of time
steps between two outputs: the steps, then the fields read back.

Families:
  run       fixed-dt steps (fen_ns_run), then u, v, (w,) p on the host
  cfl       constant CFL, one call per step, dt and maxCFL read every step
  rt        two-phase steps (Rayleigh-Taylor), then u, v, p and the vof
  adjoint   recorded forward run and the gradient of its final velocity
  poisson   one direct Poisson solve of a host array

The spacing is a power of two wherever a direction is tridiagonal: the
singular column's last pivot is then exactly zero, as its algebra says, and
the pressure's constant is not left to round-off.

`exact` restates the scheme in torch FP64 with other algorithms (dense cosine
transforms, torch's FFT, automatic differentiation for the adjoint).
"""
import math

import numpy as np
import torch

from fen_amd import Solver
from fen_amd._lib import (BC_PERIODIC, BC_WALL, FP32_REFINE, FP64, P, U, V, VOF, W)

TWO_PI = 2.0 * math.pi


def listed():
    return [
        # 2-D doubly periodic Taylor-Green vortex at the benchmark's 128^2: the smallest steps, bound by launches
        dict(name="vortex2d_128", family="run", solver="pp", nx=128, ny=128, nz=1, steps=200, fp32=False),
        # lid-driven square-ish cavity in 2-D (both directions walls); the tridiagonal direction is not a power of two
        dict(name="cavity2d_256x200", family="run", solver="nn", nx=256, ny=200, nz=1, steps=100, fp32=False),
        # the reference's Rayleigh-Taylor test, two-phase mode, at its size
        dict(name="rayleigh_taylor_128x512", family="rt", nx=128, ny=512, steps=60),
        # the reference's small 3-D convergence tests run at 16^3..64^3
        dict(name="periodic3d_32", family="run", solver="ppp", nx=32, ny=32, nz=32, steps=200, fp32=False),
        # decaying turbulence under constant CFL, the status line's numbers read every step
        dict(name="cfl_128", family="cfl", nx=128, ny=128, nz=128, steps=40, fp32=False),
        # the headline size, both forms of arithmetic
        dict(name="periodic3d_256", family="run", solver="ppp", nx=256, ny=256, nz=256, steps=200, fp32=False),
        dict(name="periodic3d_256_fp32", family="run", solver="ppp", nx=256, ny=256, nz=256, steps=200, fp32=True),
        # plane channel: long transforms in x, a ragged tridiagonal direction; the largest grid here
        dict(name="channel_512x256x192", family="run", solver="ppn", nx=512, ny=256, nz=192, steps=100, fp32=False),
        # lid-driven cavity and square duct: cosine transforms, ragged z
        dict(name="cavity3d_128x128x160", family="run", solver="nnn", nx=128, ny=128, nz=160, steps=100, fp32=False),
        dict(name="duct3d_128x256x101", family="run", solver="npn", nx=128, ny=256, nz=101, steps=100, fp32=False),
        # gradient of a recorded run at the benchmark's 128^3
        dict(name="adjoint_128", family="adjoint", nx=128, ny=128, nz=128, steps=60, every=20),
        # solve_poisson called on a host array with ghosts, as the reference's Poisson tests do
        dict(name="poisson_ppn_128x128x100", family="poisson", solver="ppn", nx=128, ny=128, nz=100, gl=1),
    ]


# A pass of a drawn run advances at most this many cells in all, a fraction of
# what the largest listed pass does.
DRAWN_CELL_STEPS = 4.0e8


def _pow2(rng, lo, hi):
    return 2 ** rng.randint(int(math.log2(lo)), int(math.log2(hi)))


def _ragged(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the listed ranges: transformed directions are powers of two
    (a condition of fen_create), tridiagonal ones any length."""
    family = rng.choice(["run", "run", "run", "run2d", "run2d", "cfl", "rt", "adjoint", "poisson"])
    if family == "run2d":
        solver = rng.choice(["pp", "pn", "nn"])
        nx, ny = _pow2(rng, 32, 512), _pow2(rng, 32, 512)
        if solver == "nn":
            ny = _ragged(rng, 24, 500)
        return dict(family="run", solver=solver, nx=nx, ny=ny, nz=1, steps=rng.randint(20, 150),
                    fp32=solver == "pp" and rng.random() < 0.3)
    if family == "rt":
        return dict(family="rt", nx=_pow2(rng, 32, 256), ny=_pow2(rng, 64, 512), steps=rng.randint(10, 60))
    if family == "adjoint":
        n = [_pow2(rng, 16, 128) for _ in range(3)]
        return dict(family="adjoint", nx=n[0], ny=n[1], nz=n[2], steps=rng.randint(8, 40), every=rng.randint(3, 20))
    if family == "poisson":
        solver = rng.choice(["pp", "pn", "nn", "ppp", "ppn", "npn", "nnn"])
        nx, ny = _pow2(rng, 16, 256), _pow2(rng, 16, 128)
        nz = 1 if len(solver) == 2 else (_pow2(rng, 16, 128) if solver == "ppp" else _ragged(rng, 10, 150))
        return dict(family="poisson", solver=solver, nx=nx, ny=ny, nz=nz, gl=rng.randint(0, 1))
    solver = "ppp" if family == "cfl" else rng.choice(["ppp", "ppn", "ppn", "npn", "nnn"])
    while True:
        nx, ny = _pow2(rng, 16, 512), _pow2(rng, 16, 256)
        nz = _pow2(rng, 16, 256) if solver == "ppp" else _ragged(rng, 9, 300)
        if nx * ny * nz <= 2 ** 23:
            break
    steps = max(5, min(100, int(DRAWN_CELL_STEPS / (nx * ny * nz)), rng.randint(20, 100)))
    if family == "cfl":
        return dict(family="cfl", nx=nx, ny=ny, nz=nz, steps=min(steps, 40), fp32=rng.random() < 0.3)
    return dict(family="run", solver=solver, nx=nx, ny=ny, nz=nz, steps=steps,
                fp32=solver in ("ppp", "ppn") and rng.random() < 0.35)


# --------------------------------------------------------------- inputs
# Fields are torch tensors with the axes reversed, f[k, j, i] (2-D: f[j, i]),
# so their memory order is the framework's (i fastest).

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Problem:
    """Grid, physics and initial interior fields of one case, from its seed."""

    def __init__(self, case, seed):
        family = case["family"]
        self.n = [case["nx"], case["ny"]] + ([case["nz"]] if case.get("nz", 1) > 1 else [])
        self.dim = len(self.n)
        self.solver = case.get("solver", {"rt": "pn"}.get(family, "ppp"))
        self.per = [c == "p" for c in self.solver]
        self.precision = FP32_REFINE if case.get("fp32") else FP64
        self.density, self.g = 1.0, [0.0, 0.0, 0.0]
        self.lid = None            # (axis, value): the high face of that axis moves along x
        nx = case["nx"]
        gen = torch.Generator(device=_device())
        gen.manual_seed(int(seed))
        self.shape = tuple(reversed(self.n))
        noise = [torch.randn(self.shape, generator=gen, device=_device(), dtype=torch.float64) for _ in range(self.dim)]
        phase = torch.rand(3, generator=gen, device=_device(), dtype=torch.float64)
        if all(self.per):
            self.delta = TWO_PI / nx
            self.nu = 0.01 if self.dim == 2 else 1.0 / 1600.0
            self.u = self._vortex(phase, noise)
            self.dt = min(0.25 * self.delta, 0.05 * self.delta ** 2 / self.nu)
        elif self.solver == "ppn":
            self.delta = 4.0 / nx
            self.nu, self.g[0], ub = 1.0 / 180.0, 1.0, 15.7
            h = 0.5 * self.n[2] * self.delta
            z = (self._axis(2) - 0.5) * self.delta / h - 1.0
            self.u = [0.05 * ub * e for e in noise]
            self.u[0] = self.u[0] + 1.5 * ub * (1.0 - z ** 2)
            self.dt = min(0.25 * self.delta / (1.5 * ub), 0.05 * self.delta ** 2 / self.nu)
        elif family == "rt":
            self.delta, self.nu, self.g[1] = 1.0 / nx, 3.13e-3, -9.80665
            self.u = [0.01 * e for e in noise]
            self.dt = None
            self.wave = 0.04 + 0.02 * float(phase[0])
        else:   # duct (npn), cavities (nn, nnn), 2-D channel (pn)
            self.delta = 1.0 / nx
            self.nu = 0.01
            self.u = [(0.05 if self.solver in ("npn", "pn") else 0.01) * e for e in noise]
            if self.solver == "npn":
                self.g[1] = 1.0
                x = (self._axis(0) - 0.5) / self.n[0]
                z = (self._axis(2) - 0.5) / self.n[2]
                self.u[1] = self.u[1] + 2.0 * 16.0 * x * (1.0 - x) * z * (1.0 - z)
            elif self.solver == "pn":
                self.g[0] = 1.0
                y = (self._axis(1) - 0.5) / self.n[1]
                self.u[0] = self.u[0] + 1.5 * 4.0 * y * (1.0 - y)
            else:
                self.lid = (self.dim - 1, 1.0)
            self.dt = min(0.2 * self.delta, 0.05 * self.delta ** 2 / self.nu)
        for a in range(self.dim):          # the normal velocity is zero on the high wall
            if not self.per[a]:
                self.u[a] = self.u[a].clone()
                self.u[a].select(self.dim - 1 - a, self.n[a] - 1).zero_()
        if self.precision != FP64:         # the FP32 form holds FP32 fields
            self.u = [f.float().double() for f in self.u]
        self.p = torch.zeros(self.shape, device=_device(), dtype=torch.float64)

    def _axis(self, a):
        x = torch.arange(1, self.n[a] + 1, device=_device(), dtype=torch.float64)
        s = [1] * self.dim
        s[self.dim - 1 - a] = -1
        return x.reshape(s)

    def _vortex(self, phase, noise):
        """Taylor-Green velocity with a seeded phase, plus noise of amplitude 1e-3."""
        c = [(self._axis(a) - 0.5) * (TWO_PI / self.n[a]) + TWO_PI * phase[a] for a in range(self.dim)]
        f = [self._axis(a) * (TWO_PI / self.n[a]) + TWO_PI * phase[a] for a in range(self.dim)]
        u, v = torch.sin(f[0]) * torch.cos(c[1]), -torch.cos(c[0]) * torch.sin(f[1])
        if self.dim == 3:
            u, v = u * torch.cos(c[2]), v * torch.cos(c[2])
        parts = [u, v] + ([torch.zeros_like(noise[2])] if self.dim == 3 else [])
        return [a + 1e-3 * e for a, e in zip(parts, noise)]

    def vof(self):
        """Interface y = Ly/2 + wave cos(2 pi x), heavy fluid above: 2x2 Gauss averages of the tanh profile."""
        d = self.delta
        r = 0.5 / math.sqrt(3.0)
        x, y = (self._axis(0) - 0.5) * d, (self._axis(1) - 0.5) * d
        f = 0.0
        for ox in (-r, r):
            for oy in (-r, r):
                dist = y + oy * d - self.wave * torch.cos(TWO_PI * (x + ox * d)) - 0.5 * self.n[1] * d
                f = f + 0.25 * 0.5 * (1.0 + torch.tanh(dist / d))
        return f


RT = dict(rho0=0.1694, rho1=1.225, mu0=3.13e-3, mu1=3.13e-3, sigma=0.0)
RT_U = 4.0   # velocity scale of set_timestep


def _host(pr, f):
    """A ghosted host array (Fortran order) with the interior f."""
    g = torch.zeros([pr.n[2] + 2 if pr.dim == 3 else 3, pr.n[1] + 2, pr.n[0] + 2], dtype=torch.float64)
    g[1:-1, 1:-1, 1:-1] = f.cpu() if pr.dim == 3 else f.cpu()[None]
    return g.numpy().T


def _make_solver(pr):
    """What a program sets up: grid, parameters, boundary values, initial fields."""
    bc = []
    for a in range(3):
        bc += [BC_PERIODIC if a >= pr.dim or pr.per[a] else BC_WALL] * 2
    n = tuple(pr.n) + ((1,) if pr.dim == 2 else ())
    s = Solver(pr.dim, n, tuple(pr.delta * m for m in n), bc=bc, precision=pr.precision)
    s.set_params(density=pr.density, viscosity=pr.nu, g=tuple(pr.g), cfl=0.5)
    if pr.lid:
        axis, value = pr.lid
        plane = np.full((n[0] + 2, (n[1] if axis == 2 else n[2]) + 2), value)
        s.set_bc_plane(U, 2 * axis + 1, plane)
    for fid, f in zip((U, V, W), pr.u):
        s.upload(fid, _host(pr, f))
        s.update_ghost_nodes(fid)
    s.upload(P, _host(pr, pr.p))
    s.update_ghost_nodes(P)
    return s


class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.case = case
    pr = _Problem(case, seed)
    st.solver = s = _make_solver(pr)
    family = case["family"]
    st.step = 0
    st.fields = [U, V, W, P] if pr.dim == 3 else [U, V, P]
    if family == "poisson":
        st.f = _poisson_input(case, pr, seed)
        return st
    if family == "rt":
        s.set_multiphase(**RT)
        s.upload(VOF, _host(pr, pr.vof()))
        s.update_ghost_nodes(VOF)
        s.update_material_properties()
        pr.dt = s.set_timestep(RT_U)
        st.fields = st.fields + [VOF]
    elif family == "cfl":
        pr.dt = s.set_timestep(2.0)
        s.set_params(density=pr.density, viscosity=pr.nu, g=tuple(pr.g), cfl=0.4, constant_cfl=True)
    else:
        s.set_dt_o(pr.dt)
    st.dt = pr.dt
    if family == "adjoint":
        # dL/d(final velocity) of a loss linear in it (a projection onto the initial flow)
        st.seed = [np.asfortranarray(f.cpu().numpy().T) for f in pr.u]
        return st
    # the host arrays the program reads its fields into
    st.host = {f: np.zeros(s.shape(f), order="F") for f in st.fields}
    if case.get("fp32"):
        # the FP32 form's fields are FP32 values: the program keeps them so
        st.out32 = {f: torch.zeros(a.T.shape, dtype=torch.float32) for f, a in st.host.items()}
    return st


NAMES = {U: "u", V: "v", W: "w", P: "p", VOF: "vof"}


def _read(st):
    """The fields into the program's host arrays (ghosts included; 2-D: the live plane)."""
    s, out = st.solver, {}
    for f, a in st.host.items():
        s._check(s.lib.fen_download(s.h, f, a.ctypes.data_as(s.lib.fen_download.argtypes[2]), a.size))
        if st.case.get("fp32"):
            st.out32[f].copy_(torch.from_numpy(a.T))
            out[NAMES[f]] = st.out32[f]
        else:
            out[NAMES[f]] = a.T
        if s.dim == 2:
            out[NAMES[f]] = out[NAMES[f]][1]
    return out


def run(st):
    case, s = st.case, st.solver
    family = case["family"]
    if family == "poisson":
        return s.solve_poisson(st.f, case["gl"]).T
    if family == "adjoint":
        s.adjoint_record(st.step, case["steps"], case["every"], st.dt)
        # (the first projection takes the initial pressure out again: no gradient to return for it)
        grads = s.adjoint_backward(st.seed)
        st.step += case["steps"]
        return [g.T for g in grads]
    if family == "cfl":
        dts, cfls = [], []
        for _ in range(case["steps"]):
            st.step += 1
            st.dt, _, cfl = s.navier_stokes_solver(st.step, st.dt)
            dts.append(st.dt)
            cfls.append(cfl)
        out = _read(st)
        # held to the fields' own type: in the FP32 form they come from FP32 fields
        kind = np.float32 if case["fp32"] else np.float64
        out["dt"], out["cfl"] = np.array(dts, kind), np.array(cfls, kind)
        return out
    s.run(st.step, case["steps"], st.dt)
    st.step += case["steps"]
    return _read(st)


def work(case):
    """A step reads the state (u, v, w, p and the last step's right-hand side)
    once and writes it once; the outputs cross to the host once."""
    cells = case["nx"] * case["ny"] * case.get("nz", 1)
    dim = 3 if case.get("nz", 1) > 1 else 2
    word = 4 if case.get("fp32") else 8
    logn = math.log2(cells)
    family = case["family"]
    solve = 5.0 * logn + 10.0                # flops per cell of transforms there and back
    if family == "poisson":
        return {"bytes": 2.0 * 8 * cells, "flops": solve * cells}
    state = 2 * dim + 1                      # u, p, dv_o
    flops = (60.0 if dim == 2 else 120.0) + solve
    steps = case["steps"]
    out = (dim + 1) * 8.0 * cells
    if family == "rt":
        return {"bytes": steps * 2.0 * (state + 2) * 8 * cells + out + 8.0 * cells, "flops": steps * (flops + 300.0) * cells}
    if family == "adjoint":
        # forward, recomputation, transposed step (the state and its adjoint)
        return {"bytes": steps * 6.0 * state * 8 * cells + 6 * 8.0 * cells, "flops": steps * 4.0 * flops * cells}
    return {"bytes": steps * 2.0 * state * word * cells + out * word / 8, "flops": steps * flops * cells}


# --------------------------------------------------------------- 64-bit values
class _Exact:
    """The scheme in torch FP64.  A ghosted field is its interior with the
    boundary rules applied along x, then y, then z over whole planes."""

    def __init__(self, pr):
        self.pr, self.dim, self.n, self.delta = pr, pr.dim, pr.n, pr.delta
        self.id = 1.0 / pr.delta
        self.dt_o = pr.dt
        dev, f64 = pr.p.device, torch.float64
        self.cos = []
        lam = torch.zeros([1] * self.dim, device=dev, dtype=f64)
        for a in range(self.dim):
            m = self.n[a]
            i = torch.arange(m, device=dev, dtype=f64)
            s = [1] * self.dim
            s[self.dim - 1 - a] = -1
            factor = TWO_PI if pr.per[a] else math.pi
            # 2 (cos t - 1) = -4 sin^2(t/2)
            lam = lam - (4.0 * torch.sin(0.5 * factor * i / m) ** 2 / pr.delta ** 2).reshape(s)
            if pr.per[a]:
                self.cos.append(None)
            else:   # orthonormal cosine basis, rows = modes
                q = torch.cos(math.pi * i[:, None] * (i[None, :] + 0.5) / m) * math.sqrt(2.0 / m)
                q[0] *= math.sqrt(0.5)
                self.cos.append(q)
        self.lam = lam

    def ax(self, a):
        return self.dim - 1 - a

    def sh(self, g, *offs):
        """The interior-shaped view of a ghosted array at an offset per axis (x first)."""
        for a, o in enumerate(offs):
            g = g.narrow(self.ax(a), 1 + o, self.n[a])
        return g

    def inner(self, g):
        return self.sh(g, *([0] * self.dim))

    def fill(self, f, comp=None):
        """comp: the velocity component (None: a centred field, Neumann at walls)."""
        pr = self.pr
        for a in range(self.dim):
            d, m = self.ax(a), self.n[a]
            first, last = f.narrow(d, 0, 1), f.narrow(d, m - 1, 1)
            if pr.per[a]:
                lo, hi = last, first
            elif comp is None:
                lo, hi = first, last
            elif comp == a:                 # impermeable wall: the faces are 0
                lo, hi = torch.zeros_like(first), torch.zeros_like(last)
                f = torch.cat([f.narrow(d, 0, m - 1), torch.zeros_like(last)], d)
            else:
                wall = pr.lid[1] if pr.lid and pr.lid[0] == a and comp == 0 else 0.0
                lo, hi = -first, 2.0 * wall - last
            f = torch.cat([lo, f, hi], d)
        return f

    def solve(self, f):
        """lap(phi) = f with the mean or the last plane's mean fixed as the solver does."""
        pr, dims = self.pr, []
        for a in range(self.dim):
            if pr.per[a]:
                dims.append(self.ax(a))
            else:
                f = torch.tensordot(f, self.cos[a], dims=([self.ax(a)], [1])).movedim(-1, self.ax(a))
        lam = torch.where(self.lam == 0.0, torch.ones_like(self.lam), self.lam)
        if dims:
            f = torch.fft.fftn(f, dim=dims)
        f = torch.where(self.lam == 0.0, torch.zeros_like(f), f / lam)
        if dims:
            f = torch.fft.ifftn(f, dim=dims).real
        for a in range(self.dim):
            if not pr.per[a]:
                f = torch.tensordot(f, self.cos[a], dims=([self.ax(a)], [0])).movedim(-1, self.ax(a))
        if pr.solver in ("nn", "npn", "nnn"):
            f = f - f[-1].mean()
        return f

    def grad(self, g, a):
        o = [0] * self.dim
        o[a] = 1
        return (self.sh(g, *o) - self.inner(g)) * self.id

    def div(self, us):
        d = 0.0
        for a in range(self.dim):
            o = [0] * self.dim
            o[a] = -1
            d = d + (self.inner(us[a]) - self.sh(us[a], *o)) * self.id
        return d

    def off(self, **k):
        o = [0] * self.dim
        for name, v in k.items():
            o[int(name[1])] += v
        return o

    def advection(self, us, a):
        r = 0.0
        for b in range(self.dim):
            at = lambda f, i=0, j=0: self.sh(us[f], *self.off(**{"a%d" % a: i, "a%d" % b: j})) if a != b else \
                self.sh(us[f], *self.off(**{"a%d" % a: i + j}))  # noqa: E731
            if a == b:
                hi, lo = 0.25 * (at(a, 1) + at(a)) ** 2, 0.25 * (at(a) + at(a, -1)) ** 2
            else:
                hi = 0.25 * (at(a, 0, 1) + at(a)) * (at(b, 1, 0) + at(b))
                lo = 0.25 * (at(a) + at(a, 0, -1)) * (at(b, 1, -1) + at(b, 0, -1))
            r = r - (hi - lo) * self.id
        return r

    def lap(self, g):
        r, c = 0.0, self.inner(g)
        for a in range(self.dim):
            k = "a%d" % a
            r = r + (self.sh(g, *self.off(**{k: 1})) - 2.0 * c + self.sh(g, *self.off(**{k: -1}))) * self.id ** 2
        return r

    def step(self, us, p, dvo, dt):
        """us, p ghosted, dvo interior; returns the next."""
        pr = self.pr
        A, B = 1.0 + 0.5 * dt / self.dt_o, -0.5 * dt / self.dt_o
        dv, star = [], []
        for a in range(self.dim):
            r = self.advection(us, a) + pr.nu / pr.density * self.lap(us[a])
            dv.append(r)
            rhs = -self.grad(p, a) / pr.density + A * r + B * dvo[a] + pr.g[a]
            star.append(self.fill(self.inner(us[a]) + dt * rhs, a))
        phi = self.fill(self.solve(self.div(star) * pr.density / dt))
        new = [self.fill(self.inner(star[a]) - dt / pr.density * self.grad(phi, a), a) for a in range(self.dim)]
        return new, self.fill(self.inner(p) + self.inner(phi)), dv

    def start(self):
        us = [self.fill(f, a) for a, f in enumerate(self.pr.u)]
        return us, self.fill(self.pr.p), [torch.zeros_like(f) for f in self.pr.u]


def _exact_rt(pr, steps):
    """The two-phase step: MTHINC advection, variable density and viscosity, constant-coefficient pressure."""
    E = _Exact(pr)
    d, small, cut, beta = pr.delta, 1e-14, 1e-8, 1.0
    rho0, rho1, mu0, mu1 = RT["rho0"], RT["rho1"], RT["mu0"], RT["mu1"]
    rmin = min(rho0, rho1)
    dt = min(0.5 * d / RT_U, 0.125 * d * d * min(rho0 / mu0, rho1 / mu1))
    E.dt_o = dt
    rp, rm = 0.5 * (1.0 + 1.0 / math.sqrt(3.0)), 0.5 * (1.0 - 1.0 / math.sqrt(3.0))

    def surface(nx, ny, lx, ly):
        cx = (nx.abs() < ny.abs()).double()
        cy = 1.0 - cx
        return cx, cy, nx - 0.5 * cx * lx, ny - 0.5 * cy * ly, 0.5 * cx * lx, 0.5 * cy * ly

    def poly(q, x, y):
        cx, cy, a10, a01, a20, a02 = q
        return cx * a20 * x * x + cy * a02 * y * y + a10 * x + a01 * y

    def reconstruct(vof):
        s = lambda i, j: E.sh(vof, i, j)  # noqa: E731
        # vertex normals, in the order (-,-), (-,+), (+,+), (+,-)
        mx = [0.5 * (s(0, b) + s(0, b + 1) - s(-1, b) - s(-1, b + 1)) / d for b in (-1, 0)]
        mx += [0.5 * (s(1, b) + s(1, b + 1) - s(0, b) - s(0, b + 1)) / d for b in (0, -1)]
        my = [0.5 * (s(-1, b + 1) + s(0, b + 1) - s(-1, b) - s(0, b)) / d for b in (-1, 0)]
        my += [0.5 * (s(0, b + 1) + s(1, b + 1) - s(0, b) - s(1, b)) / d for b in (0, -1)]
        unit = [torch.sqrt(a * a + b * b + small) for a, b in zip(mx, my)]
        nxs, nys = [a / m for a, m in zip(mx, unit)], [a / m for a, m in zip(my, unit)]
        cx, cy = 0.25 * sum(mx), 0.25 * sum(my)
        m = torch.sqrt(cx * cx + cy * cy + small)
        nx, ny = cx / m, cy / m
        lx, ly = 0.5 * d * (nxs[3] + nxs[2] - nxs[1] - nxs[0]), 0.5 * d * (nys[1] + nys[2] - nys[0] - nys[3])
        f = E.inner(vof)
        mixed = (f > cut) & (f < 1.0 - cut)
        q = surface(nx, ny, lx, ly)
        main = torch.where(q[0] == 0.0, q[2], q[3])
        pp = torch.where(q[0] == 0.0, poly(q, 0.0, rp), poly(q, rp, 0.0))
        pm = torch.where(q[0] == 0.0, poly(q, 0.0, rm), poly(q, rm, 0.0))
        a_, bp, bm = torch.exp(2 * beta * main), torch.exp(2 * beta * pp), torch.exp(2 * beta * pm)
        qq = torch.exp(2 * beta * main * (2.0 * f - 1.0))
        aa, bb, cc = a_ * bm * bp * (a_ - qq), a_ * (bp + bm) * (1.0 - qq), 1.0 - a_ * qq
        root = torch.sqrt(bb * bb - 4.0 * aa * cc)
        dd = torch.log(torch.maximum((-bb + root) / (2 * aa), (-bb - root) / (2 * aa))) / (2 * beta)
        dd = torch.where(mixed, dd, torch.zeros_like(dd))
        return [E.fill(a) for a in (nx, ny, lx, ly, dd)]

    def sweep(axis, vof, rec, vel, src):
        """One directional sweep; fluxes on the high faces of every cell and on the low face of the first."""
        nx, ny, lx, ly, dd = rec
        k = E.ax(axis)
        m = E.n[axis]
        o = 1 - axis
        trim = lambda g: g.narrow(E.ax(o), 1, E.n[o])  # noqa: E731
        face = trim(vel).narrow(k, 0, m + 1)
        plus = face >= 0
        pick = lambda g: torch.where(plus, trim(g).narrow(k, 0, m + 1), trim(g).narrow(k, 1, m + 1))  # noqa: E731
        lo = torch.where(plus, 1.0 - dt * face / d, torch.zeros_like(face))
        hi = torch.where(plus, torch.ones_like(face), -dt * face / d)
        f, d0 = pick(vof), pick(dd)
        q = surface(pick(nx), pick(ny), pick(lx), pick(ly))
        zero, one = torch.zeros_like(lo), torch.ones_like(lo)
        xa, xb, ya, yb = (lo, hi, zero, one) if axis == 0 else (zero, one, lo, hi)
        first = q[0] == 0.0     # integrate analytically along x, by two points along y
        cosh = lambda x, y: torch.cosh(beta * (poly(q, x, y) + d0))  # noqa: E731
        val = torch.zeros_like(lo)
        for r in (rm, rp):
            gx = 0.5 * (xb - xa + 1.0 / (q[2] * beta) * torch.log(cosh(xb, r * (ya + yb)) / cosh(xa, r * (ya + yb))))
            gy = 0.5 * (yb - ya + 1.0 / (q[3] * beta) * torch.log(cosh(r * (xa + xb), yb) / cosh(r * (xa + xb), ya)))
            val = val + torch.where(first, 0.5 * gx * (yb - ya), 0.5 * gy * (xb - xa))
        full = f * (xb - xa) * (yb - ya)
        val = torch.where((f > cut) & (f < 1.0 - cut), val, full)
        flux = torch.where(plus, val, -val) * d
        du = face.narrow(k, 1, m) - face.narrow(k, 0, m)
        return (E.inner(src) - (flux.narrow(k, 1, m) - flux.narrow(k, 0, m)) / d) / (1.0 - dt * du / d)

    us, p, dvo = E.start()
    vof, p_o = E.fill(pr.vof()), torch.zeros_like(p)
    order = (0, 1)
    for _ in range(steps):
        v1 = sweep(order[0], vof, reconstruct(vof), us[order[0]], vof)
        g1 = E.fill(v1)
        v2 = sweep(order[1], g1, reconstruct(g1), us[order[1]], g1)
        du = [E.inner(us[a]) - E.sh(us[a], *[-1 if b == a else 0 for b in range(2)]) for a in range(2)]
        vof = E.fill(v2 - dt / d * (v1 * du[order[0]] + v2 * du[order[1]]))
        order = order[::-1]
        rho, mu = rho1 * vof + rho0 * (1.0 - vof), mu1 * vof + mu0 * (1.0 - vof)
        p_hat = E.fill(E.inner(2.0 * p - p_o))
        dv, star = [], []
        A, B = 1.5, -0.5
        for a in range(2):
            b = 1 - a
            o = lambda i, j: (i, j) if a == 0 else (j, i)  # noqa: E731
            sa = lambda g, i, j: E.sh(g, *o(i, j))  # noqa: E731   i along a, j across
            rf = 0.5 * (sa(rho, 1, 0) + sa(rho, 0, 0))
            ua, ub = us[a], us[b]
            taa = 2.0 * (sa(mu, 1, 0) * (sa(ua, 1, 0) - sa(ua, 0, 0)) - sa(mu, 0, 0) * (sa(ua, 0, 0) - sa(ua, -1, 0)))
            tab = []
            for j in (0, -1):
                m = 0.25 * (sa(mu, 0, j) + sa(mu, 1, j) + sa(mu, 0, j + 1) + sa(mu, 1, j + 1))
                tab.append(m * (sa(ua, 0, j + 1) - sa(ua, 0, j) + sa(ub, 1, j) - sa(ub, 0, j)))
            r = E.advection(us, a) + (taa + tab[0] - tab[1]) / (d * d) / rf
            dv.append(r)
            rhs = A * r + B * dvo[a] + pr.g[a] - E.grad(p, a) / rmin - (1.0 / rf - 1.0 / rmin) * E.grad(p_hat, a)
            star.append(E.fill(E.inner(ua) + dt * rhs, a))
        dvo = dv
        phi = E.fill(E.solve(E.div(star) * rmin / dt))
        us = [E.fill(E.inner(star[a]) - dt / rmin * E.grad(phi, a), a) for a in range(2)]
        p_o, p = p, E.fill(E.inner(p) + E.inner(phi))
    return {"u": us[0], "v": us[1], "p": p, "vof": vof}


def _exact_adjoint(pr, case, seed_fields):
    """Reverse differentiation step by step: the states are kept, one step's graph at a time."""
    E = _Exact(pr)
    inner = [f.clone() for f in pr.u]
    p, dvo = pr.p.clone(), [torch.zeros_like(f) for f in pr.u]

    def one(u, p, dvo):
        us, pg, dv = E.step([E.fill(f, a) for a, f in enumerate(u)], E.fill(p), dvo, pr.dt)
        return [E.inner(f) for f in us], E.inner(pg), dv

    states = []
    for _ in range(case["steps"]):
        states.append((inner, p, dvo))
        inner, p, dvo = one(inner, p, dvo)
    bar = [f.clone() for f in seed_fields] + [torch.zeros_like(p)] + [torch.zeros_like(p) for _ in range(3)]
    for u, p, dvo in reversed(states):
        x = [f.detach().requires_grad_(True) for f in list(u) + [p] + list(dvo)]
        y, yp, ydv = one(x[:3], x[3], x[4:])
        bar = torch.autograd.grad(list(y) + [yp] + list(ydv), x, bar, allow_unused=True)
        bar = [b if b is not None else torch.zeros_like(p) for b in bar]
    return list(bar[:3])


def _poisson_input(case, pr, seed):
    """A zero-mean right-hand side, ghosts set to values of their own."""
    f = _poisson_rhs(pr)
    if not case["gl"]:
        a = f.cpu().numpy().T
        return np.asfortranarray(a if pr.dim == 3 else a[:, :, None])
    return np.asfortranarray(_host(pr, f))


def _poisson_rhs(pr):
    f = pr.u[0] + torch.sin(0.1 * pr.u[1])
    return f - f.mean()


def _exact_poisson(pr, case):
    E = _Exact(pr)
    f = E.solve(_poisson_rhs(pr))
    if not case["gl"]:
        return f if pr.dim == 3 else f[None]
    # ghosts: zero in, and the solvers that subtract a mean over the whole array shift them
    ghost = f[-1].mean() if pr.solver == "ppn" else torch.zeros((), device=f.device, dtype=f.dtype)
    full = torch.zeros([m + 2 for m in pr.shape] if pr.dim == 3 else [3] + [m + 2 for m in pr.shape],
                       device=f.device, dtype=f.dtype) + ghost
    inside = full[1:-1, 1:-1, 1:-1]
    inside.copy_(f if pr.dim == 3 else f[None])
    return full


def exact(case, seed):
    pr = _Problem(case, seed)
    family = case["family"]
    if family == "poisson":
        return _exact_poisson(pr, case)
    if family == "adjoint":
        return _exact_adjoint(pr, case, pr.u)
    with torch.no_grad():
        if family == "rt":
            return _exact_rt(pr, case["steps"])
        E = _Exact(pr)
        dts, cfls = [], []
        if family == "cfl":
            dt_visc = (1.0 / 6.0) * pr.delta ** 2 / pr.nu
            pr.dt = min(0.5 * pr.delta / 2.0, dt_visc)
            E.dt_o = pr.dt
        us, p, dvo = E.start()
        dt = pr.dt
        for _ in range(case["steps"]):
            if family == "cfl":
                speed = sum(E.inner(f).abs() for f in us).max().item()
                E.dt_o = dt
                dt = min(0.4 * pr.delta / speed, dt_visc, 1.1 * E.dt_o)
            us, p, dvo = E.step(us, p, dvo, dt)
            if family == "cfl":
                dts.append(dt)
                cfls.append(dt * sum(E.inner(f).abs() for f in us).max().item() / pr.delta)
        out = dict(zip("uvw", us))
        out["p"] = p
        if family == "cfl":
            out["dt"], out["cfl"] = np.array(dts), np.array(cfls)
        return out
