"""Kernels at the edges of their tiles and dispatch rules, against the oracle
or the plain form of the same operation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _channel(orc, nx, ny, nz, sr=3.0, nu=1 / 5600, dt=1e-3, seed=5, **kw):
    from powerllel_channel_amd import Channel
    from powerllel_channel_amd.mesh import Grid
    from powerllel_channel_amd.workloads import LX, LY, LZ
    g = Grid(nx, ny, nz, LX, LY, LZ, sr)
    G = orc.OracleGrid(nx, ny, nz, LX, LY, LZ, g.dzf, nu, dt)
    ch = Channel(nx, ny, nz, LX, LY, LZ, g.dzf, nu, dt, **kw)
    rng = np.random.default_rng(seed)
    return g, G, ch, [rng.standard_normal(g.shape) for _ in range(7)]


def _dev(torch, cuda, *arrs):
    return [torch.from_numpy(a.copy()).to(cuda) for a in arrs]


# k chunks of 1, 4 and 32 planes with a short last chunk, and of one plane on
# a grid narrower than a tile
@pytest.mark.parametrize("shape", [(64, 16, 67), (64, 256, 131), (384, 384, 33), (10, 6, 3)])
def test_stencil_chunks_bitwise(orc, cuda, shape):
    import torch
    nx, ny, nz = shape
    print(f"[stencil chunks] {shape}", flush=True)
    _, G, ch, (u, v, w, u1, v1, w1, p) = _channel(orc, nx, ny, nz)
    d = _dev(torch, cuda, u, v, w, u1, v1, w1, p)
    ch.rk1(*d[:6])
    orc.rk1(G, u, v, w, u1, v1, w1, 0.0)
    ch.rk2(*d[:6])
    orc.rk2(G, u, v, w, u1, v1, w1, 0.0)
    ch.correct_vel(d[6], *d[:3])
    orc.correct_vel(G, p, u, v, w)
    torch.cuda.synchronize()
    for a, b in zip(d[:6], (u, v, w, u1, v1, w1)):
        assert np.array_equal(a.cpu().numpy(), b)


# RK1 + RK2 in one pass (64 x 12 tiles): tiles cut by the grid's edge in x and
# y, grids narrower than the halo, k chunks of one plane and more with short
# ends, few planes
@pytest.mark.parametrize("shape,forced,u_crf,n", [
    ((4, 4, 2), (True, False, False), 0.0, 3),
    ((10, 6, 3), (True, True, False), 0.3, 4),
    ((66, 26, 17), (False, False, False), 0.2, 3),
    ((128, 24, 65), (True, False, False), 0.0, 2),
    ((256, 256, 34), (True, False, False), 0.1, 3),
    ((200, 140, 29), (False, True, False), 0.0, 4)])
def test_run_equals_steps_edges(orc, cuda, shape, forced, u_crf, n):
    """pll_channel_run against as many calls of pll_channel_step, bit for bit
    (u, v, w with their ghosts and the pressure)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    nx, ny, nz = shape
    print(f"[run = steps] {shape} forced={forced} u_crf={u_crf} n={n}", flush=True)
    g, G, ch, (u, v, w, *_) = _channel(orc, nx, ny, nz, u_crf=u_crf, is_forced=forced,
                                       vel_force=(1.0, 0.2, 0.0), dt=1e-4)
    orc.bc_vel(G, u, v, w, u_crf)
    z = np.zeros(g.shape)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    a, b = _dev(torch, cuda, u, v, w, z, z, z, z), _dev(torch, cuda, u, v, w, z, z, z, z)
    ch.run(s, n, *a)
    for _ in range(n):
        ch.step(s, *b)
    torch.cuda.synchronize()
    for q in (0, 1, 2, 6):
        assert torch.isfinite(b[q]).all()
        assert torch.equal(a[q], b[q]), q


# 64 x 4 tiles over the haloed box: sizes that fill them exactly (62 + 2 by
# 2 + 2), exceed them by one cell, and leave short k chunks
@pytest.mark.parametrize("shape", [(62, 2, 5), (63, 3, 4), (64, 6, 37), (130, 23, 16), (3, 2, 2)])
def test_rk_vjp_transposes_jvp(cuda, shape):
    """<J dq, l> = <dq, J^T l> over the haloed arrays (l on the interior), and
    the alpha, a0, beta combination.  Both sums have positive and negative
    terms of size ~1; 1e-12 of the sum of their magnitudes."""
    import torch
    from powerllel_channel_amd import Channel
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[rk vjp] {shape}", flush=True)
    g = Grid(nx, ny, nz, 0.1 * nx, 0.1 * ny, 2.0, 2.0)
    ch = Channel(nx, ny, nz, g.lx, g.ly, g.lz, g.dzf, 1e-2, 1e-3, u_crf=0.3)
    gen = torch.Generator().manual_seed(3)
    q, d, lam, x = [[torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda)
                     for _ in range(3)] for _ in range(4)]
    jd = [torch.zeros_like(t) for t in q]
    ch.rk_jvp(q, d, jd)
    o = [t.clone() for t in x]
    ch.rk_vjp(q, lam, o, 1.0, 0.0, 0.0)
    inner = (slice(1, -1),) * 3
    lhs = sum(float((a[inner] * b[inner]).sum()) for a, b in zip(jd, lam))
    rhs = sum(float((a * b).sum()) for a, b in zip(d, o))
    mag = sum(float((a * b).abs().sum()) for a, b in zip(d, o))
    assert abs(lhs - rhs) <= 1e-12 * mag
    c = [t.clone() for t in x]
    ch.rk_vjp(q, lam, c, 0.25, 1.5, -0.5)
    for a, b, l, y in zip(c, o, lam, x):
        want = 0.25 * b - 0.5 * y
        want[inner] += 1.5 * l[inner]
        assert float((a - want).abs().max()) <= 1e-14 * float(b.abs().max() + y.abs().max() + 2.0)


@pytest.mark.parametrize("shape,forced,every", [
    ((66, 18, 17), (True, False, False), 1), ((12, 10, 8), (True, True, False), 2),
    ((64, 4, 37), (False, False, True), 3), ((130, 20, 6), (False, False, False), 2)])
def test_window_gradient_vs_pieces(cuda, shape, forced, every):
    """The window's reversed steps (transposed fills, forcing and gradient
    fused into the passes around them) against the public transposes applied
    one after the other: 3 steps, 1e-11 of the largest gradient value (the
    pieces agree with the forward ones to 1e-12)."""
    import torch
    from powerllel_channel_amd import Channel, PoissonSolver
    from powerllel_channel_amd.adjoint import WallShearWindow
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[window vs pieces] {shape} forced={forced} every={every}", flush=True)
    nu, dt, n = 1e-2, 1e-3, 3
    g = Grid(nx, ny, nz, 0.1 * nx, 0.1 * ny, 2.0, 2.0)
    ch = Channel(nx, ny, nz, g.lx, g.ly, g.lz, g.dzf, nu, dt, u_crf=0.2, is_forced=forced,
                 vel_force=(1.0, 0.1, 0.0))
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    gen = torch.Generator().manual_seed(7)
    U, b = [[0.3 * torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda)
             for _ in range(3)] for _ in range(2)]
    ch.bc_vel(*U)
    win = WallShearWindow(ch, s, n, every)
    for _ in range(2):  # a second pass on the same window
        win.forward(*U, *b)
        got = [torch.full_like(U[0], 9.0) for _ in range(3)]
        win.backward(*got)
    again = [torch.zeros_like(U[0]) for _ in range(3)]
    win.backward(*again)  # and a second backward of one forward

    def zeros(m):
        return [torch.zeros_like(U[0]) for _ in range(m)]
    states, u = [], [t.clone() for t in U]
    for _ in range(n):
        states.append([t.clone() for t in u])
        ch.step_body(s, *u, *zeros(4), *b)
    inner = (slice(1, -1),) * 3
    c = nu / (n * nx * ny)

    def seed(lam):
        lam[0][1, 1:-1, 1:-1] += c / g.dzf[1]
        lam[0][nz, 1:-1, 1:-1] += c / g.dzf[nz]
    lam, grad = zeros(3), zeros(3)
    seed(lam)
    for m in range(n - 1, -1, -1):
        u1, (lp,), l1 = zeros(3), zeros(1), zeros(3)
        ch.rk1(*states[m], *u1)
        for t, f in zip(u1, b):
            t[inner] += dt * f[inner]
        ch.bc_vel(*u1)
        ch.bc_vel_adj(*lam)
        ch.force_vel_adj(*lam)
        ch.correct_vel_adj(*lam, lp)
        ch.bc_p_adj(lp)
        s.solve_adjoint(lp)
        ch.calc_rhs_adj(lp, *lam)
        ch.bc_vel_adj(*lam)
        ch.rk_vjp(u1, lam, l1, 0.5 * dt, 0.5, 0.0)
        ch.bc_vel_adj(*l1)
        for q, a, d in zip(grad, lam, l1):
            q += 0.5 * dt * a + dt * d
        ch.rk_vjp(states[m], l1, lam, dt, 1.0, 0.5)
        if m:
            seed(lam)
    top = max(float(q.abs().max()) for q in grad)
    for q, w, w2 in zip(got, grad, again):
        assert float((q - w).abs().max()) <= 1e-11 * top
        assert torch.equal(q, w2)


# z solve on ragged tiles: every rows-per-lane count with full and short last
# lanes, 2 to 64 lanes per column, plane sizes that are no multiple of a tile
# (nx ny = 24, 98 x 42, ...), tiles spanning several y rows
@pytest.mark.parametrize("shape,bc", [
    ((4, 6, 2), "NN"), ((8, 6, 9), "NN"), ((10, 14, 13), "ND"), ((24, 16, 50), "NN"),
    ((98, 42, 33), "NN"), ((36, 20, 65), "DD"), ((40, 12, 81), "NN"), ((20, 10, 127), "NN"),
    ((28, 18, 150), "NN"), ((360, 20, 180), "NN"), ((12, 30, 200), "ND"), ((60, 8, 250), "NN"),
    ((20, 12, 255), "NN"), ((24, 10, 257), "NN"), ((12, 14, 400), "NN"), ((8, 6, 512), "NN"),
    ((16, 6, 700), "NN"), ((64, 10, 1024), "NN")])
def test_ragged_z_solve(orc, cuda, shape, bc, monkeypatch):
    """The partitioned solve on ragged tiles against the oracle (1e-12, the
    solve's tolerance), its transpose against the streaming recurrence (1e-12);
    the refined form keeps the streaming solve on such grids (bit-identical)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[ragged z solve] {shape} {bc}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 3.0 if nz < 300 else 2.0)
    rng = np.random.default_rng(11)
    f = rng.standard_normal(g.shape)
    wz = g.dzf[1:-1]
    inner = (slice(1, -1),) * 3
    f[inner] -= (f[inner].sum(axis=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)

    def solver():
        return PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf, bctype_z=bc)
    monkeypatch.setenv("PLL_TRID_RAG", "1")
    rag = solver()
    monkeypatch.delenv("PLL_TRID_RAG")
    monkeypatch.setenv("PLL_TRID_STREAMING", "1")
    streaming = solver()
    monkeypatch.delenv("PLL_TRID_STREAMING")
    ref = f.copy()
    orc.OraclePPE(nx, ny, nz, g.dx, g.dy, g.dzf, bc=("PP", "PP", bc), pin_gauge=True).solve(ref)
    p, q = _dev(torch, cuda, f, f)
    rag.solve(p)
    assert np.abs(p.cpu().numpy() - ref)[inner].max() <= 1e-12 * np.abs(ref[inner]).max()
    for solve, tol in (("solve_adjoint", 1e-12), ("solve_refined", 0.0)):
        arg = (1,) if solve == "solve_refined" else ()
        p, q = _dev(torch, cuda, f, f)
        getattr(rag, solve)(p, *arg)
        getattr(streaming, solve)(q, *arg)
        a, b = p[inner], q[inner]
        assert float((a - b).abs().max()) <= tol * float(b.abs().max()), solve
        assert torch.equal(p[0], torch.from_numpy(f[0]).to(cuda))


# transform plans: every points-per-thread choice of the runtime plans (3, 4, 5,
# 7, 12; stages in registers and through LDS; rows that leave lanes of the last
# wavefront idle) and the compile-time lengths 32, 48, 96 in x and y
@pytest.mark.parametrize("shape", [
    (72, 54, 6), (216, 108, 4), (240, 120, 4), (288, 144, 4), (450, 100, 3), (24, 96, 8),
    (192, 48, 5), (96, 32, 5), (64, 140, 4), (98, 210, 3), (220, 26, 4), (432, 216, 3)])
def test_transform_plans(orc, cuda, shape):
    """Solve against the oracle (1e-12) and the refined form with two sweeps
    (1e-11, its bar)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[transform plans] {shape}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 1.0)
    f = np.random.default_rng(13).standard_normal(g.shape)
    wz = g.dzf[1:-1]
    inner = (slice(1, -1),) * 3
    f[inner] -= (f[inner].sum(axis=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)
    ref = f.copy()
    orc.OraclePPE(nx, ny, nz, g.dx, g.dy, g.dzf, pin_gauge=True).solve(ref)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    p, q = _dev(torch, cuda, f, f)
    s.solve(p)
    s.solve_refined(q, 2)
    top = np.abs(ref[inner]).max()
    assert np.abs(p.cpu().numpy() - ref)[inner].max() <= 1e-12 * top
    assert np.abs(q.cpu().numpy() - ref)[inner].max() <= 1e-11 * top


# one-pass check: rows in XCD slabs (ny a multiple of 8) and in plain order,
# fewer rows than workgroups and more, rows shorter and longer than a workgroup
@pytest.mark.parametrize("shape", [(4, 2, 2), (300, 24, 7), (20, 30, 90), (64, 128, 40)])
def test_check_equals_separate_calls(cuda, shape):
    """NaN flag, maxima and locations equal to check_nan, max_cfl, max_div; ties
    go to the first cell, NaN cells never win, infinities do."""
    import torch
    from powerllel_channel_amd import Channel
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[check] {shape}", flush=True)
    g = Grid(nx, ny, nz, 4.0, 2.0, 2.0, 2.0)
    ch = Channel(nx, ny, nz, 4.0, 2.0, 2.0, g.dzf, 1e-3, 1e-3)
    gen = torch.Generator().manual_seed(2)
    f = [torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda) for _ in range(3)]

    def compare(u, v, w):
        _, rep = ch.check(u, v, w, 1.0, 1.0)
        cfl, div = ch.max_cfl(u, v, w), ch.max_div(u, v, w)
        assert rep["nan"] == ch.check_nan(u)
        assert (rep["cfl_max"], rep["cfl_at"]) == cfl
        assert (rep["div_max"], rep["div_at"]) == div
        return rep
    assert not compare(*f)["nan"]
    const = [torch.ones_like(t) for t in f]  # every cell ties
    assert compare(*const)["cfl_at"][:2] == (1, 1)
    for at in ((0, 0, 0), (nz + 1, ny + 1, nx + 1), (1, 0, nx), (nz, ny, nx + 1), (nz, ny, nx)):
        u = f[0].clone()
        u[at] = float("nan")
        assert compare(u, *f[1:])["nan"]
    w = f[2].clone()
    w[nz, ny, 1] = float("inf")
    assert compare(f[0], f[1], w)["div_max"] == float("inf")
    everywhere = torch.full_like(f[0], float("nan"))
    assert compare(everywhere, *f[1:])["cfl_max"] == 0.0


# the corrected velocity's ghosts written by the projection: the smallest grid,
# tiles cut by the edge, k chunks with short ends
@pytest.mark.parametrize("shape,forced,u_crf", [
    ((4, 2, 2), (True, False, False), 0.3),
    ((10, 6, 3), (True, True, False), 0.3),
    ((66, 26, 17), (False, False, False), 0.2),
    ((64, 256, 131), (True, False, False), 0.0)])
def test_step_fills_boundary(orc, cuda, shape, forced, u_crf):
    """A step and a run leave the ghosts that the fill makes of their result."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    nx, ny, nz = shape
    print(f"[step fills] {shape} forced={forced}", flush=True)
    g, G, ch, (u, v, w, *_) = _channel(orc, nx, ny, nz, u_crf=u_crf, is_forced=forced,
                                       vel_force=(1.0, 0.2, 0.0), dt=1e-4)
    orc.bc_vel(G, u, v, w, u_crf)
    z = np.zeros(g.shape)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    for n in (1, 2):
        a = _dev(torch, cuda, u, v, w, z, z, z, z)
        ch.run(s, n, *a)
        b = [q.clone() for q in a[:3]]
        inner = np.full(g.shape, np.nan)
        inner[1:-1, 1:-1, 1:-1] = 0.0
        m = torch.from_numpy(inner).to(cuda)
        for q in b:
            q += m
        ch.bc_vel(*b)
        torch.cuda.synchronize()
        for x, y in zip(a[:3], b):
            assert torch.isfinite(y).all()
            assert torch.equal(x, y)


# Mean_h reduced by a workgroup of the x transform: fewer partial sums than
# threads, thread counts that are no power of two, many partial sums
@pytest.mark.parametrize("shape", [(4, 4, 2), (10, 6, 3), (66, 26, 17), (300, 140, 29),
                                   (64, 256, 131), (384, 384, 66)])
def test_forced_means(orc, cuda, shape):
    """The forcing sets Mean_h of u and v.  Their partial sums run over at most
    a few hundred terms each of size |u| <= 6 (and the pressure gradient's sum
    telescopes), so the mean is off by less than 1000 roundings of 6: 1.4e-12."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    nx, ny, nz = shape
    print(f"[forced means] {shape}", flush=True)
    g, G, ch, (u, v, w, *_) = _channel(orc, nx, ny, nz, is_forced=(True, True, False),
                                       vel_force=(1.0, 0.2, 0.0), dt=1e-4)
    orc.bc_vel(G, u, v, w, 0.0)
    z = np.zeros(g.shape)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    for n in (1, 3):
        a = _dev(torch, cuda, u, v, w, z, z, z, z)
        ch.run(s, n, *a)
        for q, m in ((a[0], 1.0), (a[1], 0.2)):
            wk = torch.from_numpy(np.asarray(g.dzf[1:-1])).to(cuda).reshape(-1, 1, 1)
            got = float((q[1:-1, 1:-1, 1:-1] * wk).sum() / wk.sum() / (nx * ny))
            assert abs(got - m) < 1.4e-12, (n, got - m)


# host-pointer solves of one chunk, two, three and five uneven ones
@pytest.mark.parametrize("shape", [(4, 4, 2), (128, 128, 97), (240, 140, 91), (192, 192, 129)])
def test_host_solve_chunks(cuda, shape):
    """The chunked host-pointer solve against the solve on the device."""
    import torch
    from powerllel_channel_amd import (PoissonSolver, execute_poisson_solver,
                                       free_poisson_solver, init_poisson_solver)
    from powerllel_channel_amd.mesh import Grid
    from powerllel_channel_amd.workloads import LX, LY, LZ
    print(f"[host chunks] {shape}", flush=True)
    g = Grid(*shape, LX, LY, LZ, 1.5)
    rhs = np.random.default_rng(3).standard_normal(g.shape)
    d = torch.from_numpy(rhs.copy()).to(cuda)
    PoissonSolver(*shape, g.dx, g.dy, g.dzf).solve(d)
    init_poisson_solver(*shape, g.dx, g.dy, g.dzf)
    try:
        for _ in range(2):
            h = rhs.copy()
            execute_poisson_solver(h)
            assert np.array_equal(h, d.cpu().numpy())
    finally:
        free_poisson_solver()


# 16-column z tiles on grids that stay in the Infinity Cache: one group per tile
# (16 rows per lane) and two (8 and 12), just above the rule's lower end
@pytest.mark.parametrize("shape", [(160, 128, 128), (96, 128, 192), (96, 96, 256), (64, 132, 256)])
def test_narrow_z_tiles(cuda, shape, monkeypatch):
    """The solve and its transpose against the streaming recurrence (1e-12, the
    solve's tolerance), the refined solve against the FP64 one (1e-9 with one
    sweep on these grids' wide tiles)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[narrow z tiles] {shape}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 2.0)
    f = np.random.default_rng(12).standard_normal(g.shape)
    wz = g.dzf[1:-1]
    inner = (slice(1, -1),) * 3
    f[inner] -= (f[inner].sum(axis=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    monkeypatch.setenv("PLL_TRID_STREAMING", "1")
    streaming = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    for solve, tol in (("solve", 1e-12), ("solve_adjoint", 1e-12), ("solve_refined", 1e-9)):
        p, q = _dev(torch, cuda, f, f)
        getattr(s, solve)(p, *((1,) if solve == "solve_refined" else ()))
        getattr(streaming, "solve" if solve == "solve_refined" else solve)(q)
        a, b = p[inner], q[inner]
        assert float((a - b).abs().max()) <= tol * float(b.abs().max()), solve


# rows per workgroup of the x transforms: the rule's 16 and 64 / T, a single row,
# counts that leave lanes of a wavefront and rows of a workgroup idle
@pytest.mark.parametrize("shape", [(4, 4, 2), (10, 6, 5), (60, 50, 21), (64, 64, 64), (96, 30, 10)])
def test_x_rows_bitwise(cuda, shape, monkeypatch):
    """The solves do not depend on the rows per workgroup."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    print(f"[x rows] {shape}", flush=True)
    g = Grid(*shape, 6.0, 3.0, 2.0, 2.0)
    f = torch.from_numpy(np.random.default_rng(13).standard_normal(g.shape)).to(cuda)
    got = []
    for rows in (None, "1", "7", "64"):
        if rows:
            monkeypatch.setenv("PLL_X_ROWS", rows)
        s = PoissonSolver(*shape, g.dx, g.dy, g.dzf)
        p, q = f.clone(), f.clone()
        s.solve(p)
        s.solve_refined(q, 1)
        got.append((p, q))
    for p, q in got[1:]:
        assert torch.equal(p, got[0][0]) and torch.equal(q, got[0][1])
