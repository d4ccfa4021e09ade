"""The adjoint window's passes on k chunks of several planes (RK1 and RK2 in one
pass with a body force, the transposed Jacobian with its carried z fluxes)."""
import pytest

pytestmark = pytest.mark.gpu


def _window(cuda, shape, forced, n, every):
    import torch
    from powerllel_channel_amd import Channel, PoissonSolver
    from powerllel_channel_amd.adjoint import WallShearWindow
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    g = Grid(nx, ny, nz, 0.1 * nx, 0.1 * ny, 2.0, 2.0)
    ch = Channel(nx, ny, nz, g.lx, g.ly, g.lz, g.dzf, 1e-2, 1e-3, u_crf=0.2, is_forced=forced,
                 vel_force=(1.0, 0.1, 0.0))
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    gen = torch.Generator().manual_seed(9)
    f = [0.3 * torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda) for _ in range(6)]
    ch.bc_vel(*f[:3])
    return ch, s, WallShearWindow(ch, s, n, every), f


# planes per chunk of the fused pass (of the partial sums) that the rules, or
# PLL_RK_KC, give: 6 (2), 2 (1), 3 without sums, 17 (17, one chunk), 8 (8, the last
# one of 7), 4 (4, the last one of 1), 3 (3), 5 (5)
@pytest.mark.parametrize("shape,forced,kc", [
    ((200, 140, 29), (True, False, False), None), ((64, 64, 64), (True, True, False), None),
    ((64, 256, 31), (False, False, False), None), ((66, 18, 17), (True, True, False), "17"),
    ((66, 26, 23), (False, True, False), "8"), ((10, 6, 9), (False, False, False), "4"),
    ((128, 24, 21), (True, False, False), "3"), ((66, 26, 30), (False, False, False), "5")])
def test_window_forward_equals_steps(cuda, shape, forced, kc, monkeypatch):
    """J of the window equals that of the same steps one by one, bit for bit."""
    import torch
    if kc:
        monkeypatch.setenv("PLL_RK_KC", kc)
    print(f"[window forward] {shape} forced={forced} kc={kc}", flush=True)
    n = 4
    ch, s, win, f = _window(cuda, shape, forced, n, 2)
    J = win.forward(*f)
    u = [t.clone() for t in f[:3]]
    tau = 0.0
    for _ in range(n):
        ch.step_body(s, *u, *[torch.zeros_like(u[0]) for _ in range(4)], *f[3:])
        tau += ch.wall_shear(u[0])
    assert torch.isfinite(u[0]).all()
    assert J == tau / n


@pytest.mark.parametrize("shape,forced", [((66, 18, 17), (True, True, False)),
                                          ((10, 6, 9), (False, False, True)),
                                          ((128, 24, 21), (False, False, False))])
def test_window_gradient_does_not_depend_on_chunks(cuda, shape, forced, monkeypatch):
    """The gradient with chunks of 2, 5 and 64 planes against chunks of one plane
    (which the small-grid tests check): 1e-11 of its largest value, the bar that
    the window's passes are held to against the separate transposes."""
    import torch
    print(f"[window gradient, chunks] {shape} forced={forced}", flush=True)
    got = []
    for kc in ("1", "2", "5", "64"):
        monkeypatch.setenv("PLL_RK_KC", kc)
        _, _, win, f = _window(cuda, shape, forced, 3, 2)
        win.forward(*f)
        grad = [torch.full_like(f[0], 9.0) for _ in range(3)]
        win.backward(*grad)
        got.append(grad)
    top = max(float(q.abs().max()) for q in got[0])
    assert top > 0.0
    for other in got[1:]:
        for a, b in zip(other, got[0]):
            assert float((a - b).abs().max()) <= 1e-11 * top


def test_window_gradient_many_planes(cuda):
    """More planes than a launch grid's z extent: the window's reversed steps
    against the public transposes applied one after the other.  The mean mode's
    pressure is summed over 65600 planes up to 65600 times its own difference
    from plane to plane, so those differences are good to some 65600 roundings,
    7e-12 of the largest; 1e-9."""
    import torch
    from powerllel_channel_amd import Channel, PoissonSolver
    from powerllel_channel_amd.adjoint import WallShearWindow
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz, nu, dt, n = 4, 2, 65600, 1e-2, 1e-3, 2
    print(f"[window gradient] {(nx, ny, nz)}", flush=True)
    g = Grid(nx, ny, nz, 0.1 * nx, 0.1 * ny, 0.1 * nz, 0.0)
    ch = Channel(nx, ny, nz, g.lx, g.ly, g.lz, g.dzf, nu, dt, is_forced=(False, False, False))
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    gen = torch.Generator().manual_seed(6)
    f = [0.3 * torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda) for _ in range(6)]
    ch.bc_vel(*f[:3])
    win = WallShearWindow(ch, s, n, 1)
    win.forward(*f)
    got = [torch.full_like(f[0], 9.0) for _ in range(3)]
    win.backward(*got)

    def zeros(m):
        return [torch.zeros_like(f[0]) for _ in range(m)]

    def seed(lam):
        for k in (1, nz):
            lam[0][k, 1:-1, 1:-1] += nu / (n * nx * ny) / g.dzf[k]
    inner = (slice(1, -1),) * 3
    second = [t.clone() for t in f[:3]]
    ch.step_body(s, *second, *zeros(4), *f[3:])
    lam, grad = zeros(3), zeros(3)
    seed(lam)
    for state in (second, f[:3]):
        u1, (lp,), l1 = zeros(3), zeros(1), zeros(3)
        ch.rk1(*state, *u1)
        for t, b in zip(u1, f[3:]):
            t[inner] += dt * b[inner]
        ch.bc_vel(*u1)
        ch.bc_vel_adj(*lam)
        ch.correct_vel_adj(*lam, lp)
        ch.bc_p_adj(lp)
        s.solve_adjoint(lp)
        ch.calc_rhs_adj(lp, *lam)
        ch.bc_vel_adj(*lam)
        ch.rk_vjp(u1, lam, l1, 0.5 * dt, 0.5, 0.0)
        ch.bc_vel_adj(*l1)
        for q, a, d in zip(grad, lam, l1):
            q += 0.5 * dt * a + dt * d
        ch.rk_vjp(state, l1, lam, dt, 1.0, 0.5)
        seed(lam)
    for q, want in zip(got, grad):
        top = float(want.abs().max())
        assert float(want[65540:, 1:-1, 1:-1].abs().max()) > 0.01 * top > 0.0
        assert float((q - want).abs().max()) <= 1e-9 * top
