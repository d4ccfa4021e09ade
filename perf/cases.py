"""Performance cases of the channel-flow hot path, run through the public API.

Kinds of case (the "kind" entry):

  solve    one pressure Poisson solve on a device array (PoissonSolver.solve)
  refined  the same solve in FP32 with FP64-residual sweeps (solve_refined)
  host     the drop-in call on a host array (execute_poisson_solver), the
           call pattern of the Fortran main program
  run      time steps (Channel.run; one step: Channel.step)
  check    the run-time checks and wall monitors between steps
  adjoint  gradient of the mean wall shear over a window of steps

Flow cases use the channel 4 pi x 2 pi x 2 of the workloads (lengths in half
heights).  Solver cases use the same box in full heights, 2 pi x pi x 1, whose
operator has no eigenvalue below 1, so a program may keep solving in place.
"""
import math

import numpy as np
import torch

FLOW_BOX = (4.0 * math.pi, 2.0 * math.pi, 2.0)
SOLVE_BOX = (2.0 * math.pi, math.pi, 1.0)


def listed():
    return [
        # Smallest solve: a test grid, where launches and latency are the cost.
        _solve("solve_64x64x64", 64, 64, 64, 1.5),
        # A grid that is no power of two in any direction (x 2^3 3^2 5,
        # y 2^3 5^2, z 2 3 5^2), as a user picks it for a resolution and not
        # for the transforms.
        _solve("solve_360x200x150", 360, 200, 150, 1.5),
        # The solver benchmark's grid, FP64 and with one refinement sweep.
        _solve("solve_768x384x256", 768, 384, 256, 2.0),
        _solve("refined_768x384x256", 768, 384, 256, 2.0, kind="refined", sweeps=1),
        # The drop-in call from a CPU program: the array crosses PCIe both ways.
        _solve("host_192x192x128", 192, 192, 128, 1.5, kind="host"),
        # One step of the smallest workload (a program that looks at its
        # fields after each step).
        _run("step_64x64x64", 64, 64, 64, 1.5, 1.0 / 5600, 1e-3, 1),
        # Ten steps between two outputs: the Re_tau 180 type of workload.
        _run("run_192x192x128", 192, 192, 128, 1.5, 1.0 / 5600, 5e-4, 10),
        # Ten steps on a grid of odd lengths.
        _run("run_240x140x90", 240, 140, 90, 1.5, 1.0 / 5600, 5e-4, 10),
        # Steps of the benchmark's grid and of the largest workload.
        _run("run_768x384x256", 768, 384, 256, 2.0, 1.0 / 5600, 1e-4, 5),
        _run("run_1536x1024x384", 1536, 1024, 384, 2.2, 1.0 / 40000, 1e-4, 3),
        # The checks of the time loop (NaN, CFL, divergence) with the wall
        # monitors, every nt_check steps of a run.
        dict(name="check_768x384x256", kind="check", nx=768, ny=384, nz=256, gamma=2.0,
             nu=1.0 / 5600, dt=1e-4),
        # Gradient of the wall shear: the differentiable workload.
        dict(name="adjoint_256x192x128", kind="adjoint", nx=256, ny=192, nz=128, gamma=1.5,
             nu=1.0 / 10000, dt=2e-4, steps=20, every=5),
    ]


def _solve(name, nx, ny, nz, gamma, kind="solve", sweeps=-1):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, gamma=gamma, sweeps=sweeps)


def _run(name, nx, ny, nz, gamma, nu, dt, steps):
    return dict(name=name, kind="run", nx=nx, ny=ny, nz=nz, gamma=gamma, nu=nu, dt=dt, steps=steps)


def draw(rng):
    """One more case.  x and y lengths are even with prime factors up to 7 (a
    few with 11 or 13), z lengths are any number."""
    kind = rng.choice(["solve", "solve", "refined", "run", "run", "run", "check", "adjoint"])
    if kind == "adjoint":
        top = (160, 128, 96)
    elif kind == "run":
        top = (640, 384, 256)
    else:
        top = (768, 512, 320)
    nx, ny = _length(rng, 24, top[0]), _length(rng, 16, top[1])
    nz = round(math.exp(rng.uniform(math.log(12), math.log(top[2]))))
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, gamma=rng.choice([0.0, 1.0, 1.5, 2.0]))
    if kind in ("solve", "refined"):
        case["sweeps"] = rng.choice([1, 2]) if kind == "refined" else -1
        return case
    case["nu"] = rng.choice([1.0 / 2000, 1.0 / 5600, 1.0 / 10000])
    dzm = float(_dzf(nz, 2.0, case["gamma"]).min())
    case["dt"] = min(0.05 * FLOW_BOX[0] / nx, 0.05 * FLOW_BOX[1] / ny, 0.2 * dzm,
                     0.1 * dzm * dzm / case["nu"], 2e-3)
    if kind == "run":
        case["steps"] = rng.choice([1, 1, 3, 5, 8])
    if kind == "adjoint":
        case["steps"] = rng.choice([2, 5, 8])
        case["every"] = rng.choice([2, 3, 8])
    return case


def _length(rng, lo, hi):
    n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    primes = (2, 3, 5, 7, 11, 13) if rng.random() < 0.15 else (2, 3, 5, 7)
    while n > lo:
        m = n // 2 if n % 2 == 0 else 0
        r = m
        for p in primes:
            while r and r % p == 0:
                r //= p
        if r == 1 and (m % 2 == 0 or len(primes) == 4):
            return n
        n -= 1
    return lo


# ------------------------------------------------------------------ inputs
def _dzf(nz, lz, gamma):
    """Cell heights of the tanh-stretched mesh with one ghost at both ends."""
    if gamma == 0.0:
        return np.full(nz + 2, lz / nz)
    s = 2.0 * gamma
    zf = [0.5 * (1.0 + math.tanh((k / nz - 0.5) * s) / math.tanh(0.5 * s)) for k in range(nz + 1)]
    zf[0] = 0.0
    d = [lz * (zf[k + 1] - zf[k]) for k in range(nz)]
    return np.array([d[0]] + d + [d[-1]])


def _rhs(case, seed):
    """Haloed right-hand side with zero ghosts: noise whose amplitude falls
    like a velocity spectrum in (kx, ky), white in z, without mean."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    gen = torch.Generator("cuda").manual_seed(seed)
    kx = torch.arange(nx // 2 + 1, device="cuda", dtype=torch.float64)
    ky = torch.fft.fftfreq(ny, 1.0 / ny, device="cuda", dtype=torch.float64) * 2.0
    amp = (1.0 + kx[None, :] ** 2 + ky[:, None] ** 2) ** (-5.0 / 6.0)
    p = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
    for k0 in range(0, nz, 32):
        n = min(32, nz - k0)
        f = torch.randn((n, ny, nx), generator=gen, dtype=torch.float64, device="cuda")
        p[1 + k0:1 + k0 + n, 1:-1, 1:-1] = torch.fft.irfft2(torch.fft.rfft2(f) * amp, s=(ny, nx))
    wz = torch.as_tensor(_dzf(nz, SOLVE_BOX[2], case["gamma"])[1:-1], device="cuda")
    inner = p[1:-1, 1:-1, 1:-1]
    inner -= (inner.sum(dim=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)
    return p


def _fields(case, seed):
    """Haloed u, v, w with zero ghosts: a laminar profile with noise."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    gen = torch.Generator("cuda").manual_seed(seed)
    dzf = _dzf(nz, FLOW_BOX[2], case["gamma"])
    z = np.cumsum(dzf[1:-1]) - 0.5 * dzf[1:-1] - 1.0
    prof = torch.as_tensor(1.5 * (1.0 - z * z), device="cuda")
    out = []
    for f in range(3):
        q = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
        inner = q[1:-1, 1:-1, 1:-1]
        inner.copy_(torch.rand((nz, ny, nx), generator=gen, dtype=torch.float64, device="cuda"))
        inner.mul_(0.2).sub_(0.1)
        if f == 0:
            inner.add_(prof[:, None, None])
        out.append(q)
    return out


def _body(case, seed):
    """Body force: small noise over the whole haloed arrays."""
    shape = (case["nz"] + 2, case["ny"] + 2, case["nx"] + 2)
    gen = torch.Generator("cuda").manual_seed(seed + 1)
    return [1e-3 * torch.randn(shape, generator=gen, dtype=torch.float64, device="cuda")
            for _ in range(3)]


def _make_solver(case, box):
    from powerllel_channel_amd import PoissonSolver
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return PoissonSolver(nx, ny, nz, box[0] / nx, box[1] / ny, _dzf(nz, box[2], case["gamma"]))


def _make_channel(case):
    from powerllel_channel_amd import Channel
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return Channel(nx, ny, nz, *FLOW_BOX, _dzf(nz, FLOW_BOX[2], case["gamma"]), case["nu"],
                   case["dt"])


_host_grid = None  # the drop-in has one instance; its grid is that of the last host case


def prepare(case, seed):
    global _host_grid
    kind = case["kind"]
    st = dict(case)
    if kind in ("solve", "refined"):
        st["solver"] = _make_solver(case, SOLVE_BOX)
        st["p"] = _rhs(case, seed)
    elif kind == "host":
        from powerllel_channel_amd import free_poisson_solver, init_poisson_solver
        grid = (case["nx"], case["ny"], case["nz"], case["gamma"])
        if _host_grid != grid:
            if _host_grid is not None:
                free_poisson_solver()
            init_poisson_solver(*grid[:3], SOLVE_BOX[0] / grid[0], SOLVE_BOX[1] / grid[1],
                                _dzf(grid[2], SOLVE_BOX[2], grid[3]))
            _host_grid = grid
        st["p"] = _rhs(case, seed).cpu().numpy()
    else:
        ch = st["channel"] = _make_channel(case)
        st["u"], st["v"], st["w"] = _fields(case, seed)
        ch.bc_vel(st["u"], st["v"], st["w"])
        if kind != "check":
            st["solver"] = _make_solver(case, FLOW_BOX)
        if kind == "run":
            for q in ("u1", "v1", "w1", "p"):
                st[q] = torch.zeros_like(st["u"])
        if kind == "adjoint":
            from powerllel_channel_amd.adjoint import WallShearWindow
            st["window"] = WallShearWindow(ch, st["solver"], case["steps"], case["every"])
            st["body"] = [b.requires_grad_() for b in _body(case, seed)]
    torch.cuda.synchronize()
    return st


def run(state):
    kind = state["kind"]
    if kind == "solve":
        state["solver"].solve(state["p"])
        return state["p"]
    if kind == "refined":
        state["solver"].solve_refined(state["p"], state["sweeps"])
        return state["p"]
    if kind == "host":
        from powerllel_channel_amd import execute_poisson_solver
        execute_poisson_solver(state["p"])
        return state["p"]
    ch, u, v, w = state["channel"], state["u"], state["v"], state["w"]
    if kind == "run":
        rest = (u, v, w, state["u1"], state["v1"], state["w1"], state["p"])
        if state["steps"] == 1:
            ch.step(state["solver"], *rest)
        else:
            ch.run(state["solver"], state["steps"], *rest)
        return [u, v, w, state["p"]]
    if kind == "check":
        _, rep = ch.check(u, v, w, 1.0, 1e-8)
        (ub, cb), (ut, ct) = ch.skin_friction(u)
        return [int(rep["nan"]), rep["cfl_max"], *rep["cfl_at"], rep["div_max"], *rep["div_at"],
                ub, cb, ut, ct, ch.mean_h(u)]
    from powerllel_channel_amd.adjoint import wall_shear_objective
    J = wall_shear_objective(state["window"], u, v, w, *state["body"])
    return [J.detach(), *torch.autograd.grad(J, state["body"])]


# ------------------------------------------------------------------ work
def work(case):
    """Inputs read once and outputs written once: the solve's array; u, v, w
    of every step and its pressure; the three fields of a check; states, body
    force and gradient of an adjoint window (forward and backward)."""
    nx, ny, nz, kind = case["nx"], case["ny"], case["nz"], case["kind"]
    n = nx * ny * nz
    solve = n * (5.0 * math.log2(nx) + 5.0 * math.log2(ny) + 8.0)
    if kind in ("solve", "host"):
        return {"bytes": 16.0 * n, "flops": solve}
    if kind == "refined":
        return {"bytes": 16.0 * n, "flops": (1 + case["sweeps"]) * solve + 20.0 * n * case["sweeps"]}
    step = 2 * 190.0 * n + solve + 20.0 * n
    if kind == "run":
        return {"bytes": 56.0 * n * case["steps"], "flops": step * case["steps"]}
    if kind == "check":
        return {"bytes": 24.0 * n, "flops": 22.0 * n}
    s = case["steps"]
    return {"bytes": 56.0 * n * s + 104.0 * n * s + 48.0 * n, "flops": 4.0 * step * s}


# ------------------------------------------------------------------ exact values
class _Reference:
    """The discrete equations in plain torch, FP64, on interior arrays
    (nz, ny, nx); the few z systems close to singular are solved in long
    double."""

    def __init__(self, case, box):
        self.nx, self.ny, self.nz = case["nx"], case["ny"], case["nz"]
        self.hx, self.hy = box[0] / self.nx, box[1] / self.ny
        self.nu, self.dt = case.get("nu", 0.0), case.get("dt", 1.0)
        d = self.dzf = _dzf(self.nz, box[2], case["gamma"])
        a = 2.0 / (d[1:-1] * (d[:-2] + d[1:-1]))
        c = 2.0 / (d[1:-1] * (d[2:] + d[1:-1]))
        b = -a - c
        b[0] += a[0]
        b[-1] += c[-1]
        a[0] = c[-1] = 0.0
        self.a, self.b, self.c = a, b, c
        self.aT = np.concatenate([[0.0], c[:-1]])
        self.cT = np.concatenate([a[1:], [0.0]])
        lx = [2.0 * (math.cos(2.0 * math.pi * i / self.nx) - 1.0) / (self.hx * self.hx)
              for i in range(self.nx // 2 + 1)]
        ly = [2.0 * (math.cos(2.0 * math.pi * i / self.ny) - 1.0) / (self.hy * self.hy)
              for i in range(self.ny)]
        self.lam = np.array(ly)[:, None] + np.array(lx)[None, :]
        col = lambda q: torch.as_tensor(q, device="cuda")[:, None, None]  # noqa: E731
        self.dz, self.dzi = col(d), col(1.0 / d)
        self.dci = col(1.0 / (0.5 * (d[:-1] + d[1:])))  # between planes k and k + 1
        self.wz = col(d[1:-1] / box[2])

    def solve(self, f, transposed=False):
        a, c = (self.aT, self.cT) if transposed else (self.a, self.c)
        F = torch.fft.rfft2(f)
        lam = torch.as_tensor(self.lam, device="cuda")
        low = np.argwhere(np.abs(self.lam) < 1e-3 * np.abs(self.b).max())
        low = low[np.argsort(np.abs(self.lam[low[:, 0], low[:, 1]]))[:2000]]
        jl, il = torch.as_tensor(low[:, 0], device="cuda"), torch.as_tensor(low[:, 1], device="cuda")
        D = F[:, jl, il].cpu().numpy().astype(np.clongdouble)
        self._thomas(D, self.lam[low[:, 0], low[:, 1]].astype(np.longdouble), a, c,
                     np.flatnonzero((low == 0).all(axis=1)))
        self._thomas(F, lam, a, c, None)
        F[:, jl, il] = torch.as_tensor(D.astype(np.complex128), device="cuda")
        return torch.fft.irfft2(F, s=(self.ny, self.nx))

    def _thomas(self, F, lam, a, c, pinned):
        b, n = self.b, self.nz
        piv = [b[0] + lam]
        for k in range(1, n):
            m = a[k] / piv[-1]
            piv.append((b[k] + lam) - m * c[k - 1])
            F[k] -= m * F[k - 1]
        F[n - 1] /= piv[-1]
        if pinned is not None:
            F[n - 1, pinned] = 0.0  # the constant of the pressure
        for k in range(n - 2, -1, -1):
            F[k] = (F[k] - c[k] * F[k + 1]) / piv[k]

    @staticmethod
    def walls(u, v, w):
        """z ghosts: no slip for u and v; w is zero on both walls."""
        zero = torch.zeros_like(w[:1])
        return (torch.cat([-u[:1], u, -u[-1:]]), torch.cat([-v[:1], v, -v[-1:]]),
                torch.cat([zero, w[:-1], zero, zero]))

    def momentum(self, u, v, w):
        xp, xm = (lambda q: torch.roll(q, -1, 2)), (lambda q: torch.roll(q, 1, 2))
        yp, ym = (lambda q: torch.roll(q, -1, 1)), (lambda q: torch.roll(q, 1, 1))
        ix, iy = 1.0 / self.hx, 1.0 / self.hy
        ct, cb = self.dci[1:], self.dci[:-1]  # above and below the cell centre
        kz = self.dzi[1:-1]
        C, P, M = (lambda q: q[1:-1]), (lambda q: q[2:]), (lambda q: q[:-2])

        def top(q):  # q at the face above
            return (C(q) * self.dz[2:] + P(q) * self.dz[1:-1]) * ct

        def bottom(q):
            return (C(q) * self.dz[:-2] + M(q) * self.dz[1:-1]) * cb

        def lap(q, up, dn, mid):
            c = C(q)
            return self.nu * ((xp(c) - 2.0 * c + xm(c)) * (ix * ix)
                              + (yp(c) - 2.0 * c + ym(c)) * (iy * iy)
                              + ((P(q) - c) * up - (c - M(q)) * dn) * mid)

        uc, vc, wc, wm = C(u), C(v), C(w), M(w)
        ue, un, vn = uc + xp(uc), uc + yp(uc), vc + yp(vc)
        ve = vc + xp(vc)
        conv = (ue * ue - xm(ue * ue)) * ix + (un * ve - ym(un * ve)) * iy \
            + (top(u) * (wc + xp(wc)) - bottom(u) * (wm + xp(wm))) * kz
        fu = lap(u, ct, cb, kz) - 0.25 * conv
        conv = (un * ve - xm(un * ve)) * ix + (vn * vn - ym(vn * vn)) * iy \
            + (top(v) * (wc + yp(wc)) - bottom(v) * (wm + yp(wm))) * kz
        fv = lap(v, ct, cb, kz) - 0.25 * conv
        ut, vt = top(u) * (wc + xp(wc)), top(v) * (wc + yp(wc))
        wt, wb = wc + P(w), wc + wm
        conv = (ut - xm(ut)) * ix + (vt - ym(vt)) * iy + (wt * wt - wb * wb) * ct
        fw = lap(w, self.dzi[2:], kz, ct) - 0.25 * conv
        return fu, fv, fw

    def step(self, u, v, w, body=(0.0, 0.0, 0.0), solve=None):
        dt = self.dt
        f = self.momentum(*self.walls(u, v, w))
        s = [q + dt * (r + b) for q, r, b in zip((u, v, w), f, body)]
        f = self.momentum(*self.walls(*s))
        g = self.walls(*s)
        u, v, w = [(q[1:-1] + dt * (r + b) + o) * 0.5
                   for q, r, b, o in zip(g, f, body, (u, v, w))]
        w = torch.cat([w[:-1], torch.zeros_like(w[:1])])
        wb = torch.cat([torch.zeros_like(w[:1]), w[:-1]])
        div = (u - torch.roll(u, 1, 2)) / self.hx + (v - torch.roll(v, 1, 1)) / self.hy \
            + (w - wb) * self.dzi[1:-1]
        p = (solve or self.solve)(div / dt)
        u = u - (torch.roll(p, -1, 2) - p) * (dt / self.hx)
        v = v - (torch.roll(p, -1, 1) - p) * (dt / self.hy)
        w = w - (torch.cat([p[1:], p[-1:]]) - p) * (dt * self.dci[1:])
        u = u + (1.0 - (u * self.wz).sum() / (self.nx * self.ny))
        return u, v, w, p

    def shear(self, u):
        n = self.nx * self.ny
        return [self.nu * u[k].sum() / n / (0.5 * self.dzf[g]) for k, g in ((0, 1), (-1, -2))]


def _halo(q):
    """Periodic ghosts in x and y of an array that has its z ghosts."""
    q = torch.cat([q[:, -1:], q, q[:, :1]], dim=1)
    return torch.cat([q[:, :, -1:], q, q[:, :, :1]], dim=2)


def _inner(q):
    return q[1:-1, 1:-1, 1:-1].contiguous()


def exact(case, seed):
    if case["nx"] * case["ny"] * case["nz"] > 10 ** 8:
        return None
    kind = case["kind"]
    if kind in ("solve", "refined", "host"):
        p = _rhs(case, seed)
        p[1:-1, 1:-1, 1:-1] = _Reference(case, SOLVE_BOX).solve(_inner(p))
        return p.cpu().numpy() if kind == "host" else p
    ref = _Reference(case, FLOW_BOX)
    u, v, w = (_inner(q) for q in _fields(case, seed))
    if kind == "check":
        return _exact_check(case, ref, u, v, w)
    w[-1] = 0.0
    if kind == "run":
        p = None
        for _ in range(case["steps"]):
            u, v, w, p = ref.step(u, v, w)
        u, v, w = ref.walls(u, v, w)
        return [_halo(q) for q in (u, v, w, torch.cat([p[:1], p, p[-1:]]))]
    return _exact_adjoint(case, ref, seed, u, v, w)


def _exact_check(case, ref, u, v, w):
    u, v, w = ref.walls(u, v, w)
    u, v, wb, w = u[1:-1], v[1:-1], w[:-2], w[1:-1]
    um, vm, dzi = torch.roll(u, 1, 2), torch.roll(v, 1, 1), ref.dzi[1:-1]
    out = [int(torch.isnan(u).any())]
    cfl = (u + um).abs() * (0.5 / ref.hx) + (v + vm).abs() * (0.5 / ref.hy) \
        + (w + wb).abs() * (0.5 * dzi)
    div = ((u - um) / ref.hx + (v - vm) / ref.hy + (w - wb) * dzi).abs()
    for q, scale in ((cfl, case["dt"]), (div, 1.0)):
        at = int(q.flatten().argmax())
        nx, ny = case["nx"], case["ny"]
        out += [float(q.flatten()[at]) * scale, at % nx + 1, at // nx % ny + 1,
                at // (nx * ny) + 1]
    for tau in ref.shear(u):
        out += [math.sqrt(float(tau)), 2.0 * float(tau)]
    return out + [float((u * ref.wz).sum() / (ref.nx * ref.ny))]


def _exact_adjoint(case, ref, seed, u, v, w):
    from torch.utils.checkpoint import checkpoint

    class Solve(torch.autograd.Function):
        @staticmethod
        def forward(ctx, f):
            return ref.solve(f)

        @staticmethod
        def backward(ctx, g):
            return ref.solve(g, transposed=True)

    body = [_inner(b).requires_grad_() for b in _body(case, seed)]

    def step(u, v, w, *b):
        return ref.step(u, v, w, b, Solve.apply)[:3]

    J = 0.0
    for _ in range(case["steps"]):
        u, v, w = checkpoint(step, u, v, w, *body, use_reentrant=False)
        tb, tt = ref.shear(u)
        J = J + 0.5 * (tb + tt) / case["steps"]
    pad = torch.nn.functional.pad
    return [J.detach(), *(pad(g, (1,) * 6) for g in torch.autograd.grad(J, body))]
