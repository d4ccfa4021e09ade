"""Which kernel a solve takes where several could, against a solver that is
held to one of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# nx a multiple of 4 but not of 8: FP32 sweeps on regular tiles of 4 columns (2 to
# 64 lanes per column), streaming above 24576 columns per lane; FP64 ragged
@pytest.mark.parametrize("shape,held", [
    ((20, 12, 16), "PLL_TRID_RAG=0"), ((12, 14, 48), "PLL_TRID_RAG=0"),
    ((100, 10, 64), "PLL_TRID_RAG=0"), ((28, 6, 96), "PLL_TRID_RAG=0"),
    ((20, 16, 128), "PLL_TRID_RAG=0"), ((12, 8, 192), "PLL_TRID_RAG=0"),
    ((36, 6, 256), "PLL_TRID_RAG=0"), ((12, 6, 512), "PLL_TRID_RAG=0"),
    ((260, 192, 16), "PLL_TRID_STREAMING=1")])
def test_refined_z_tiles_of_4_columns(cuda, shape, held, monkeypatch):
    """The refined solve is bit for bit that of a solver held to the z solve the
    rule names; the FP64 solve and its transpose agree with the streaming
    recurrence (1e-12, the solve's tolerance)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[refined, 4-column z tiles] {shape}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 2.0)
    f = np.random.default_rng(17).standard_normal(g.shape)
    wz = g.dzf[1:-1]
    inner = (slice(1, -1),) * 3
    f[inner] -= (f[inner].sum(axis=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)

    def solver(env=None):
        if env:
            monkeypatch.setenv(*env.split("="))
        s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
        if env:
            monkeypatch.delenv(env.split("=")[0])
        return s

    def run(s, name, *args):
        p = torch.from_numpy(f.copy()).to(cuda)
        getattr(s, name)(p, *args)
        return p[inner]
    default, alone, streaming = solver(), solver(held), solver("PLL_TRID_STREAMING=1")
    for sweeps in (0, 1):
        assert torch.equal(run(default, "solve_refined", sweeps),
                           run(alone, "solve_refined", sweeps)), sweeps
    for name in ("solve", "solve_adjoint"):
        a, b = run(default, name), run(streaming, name)
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max()), name


# transform plans: lengths with a factor 11 or 13 and long y transforms, at many
# threads a row (small grids), and above 2^20 cells at 12, 8, 7, 6 and 4 points per
# thread in y tiles of two columns and more, and of one
@pytest.mark.parametrize("shape", [
    (132, 66, 4), (264, 156, 3), (660, 132, 3), (252, 126, 4), (12, 1400, 3), (16, 960, 3),
    (8, 1300, 2), (132, 66, 122), (264, 156, 26), (176, 104, 58), (462, 78, 30), (660, 132, 13),
    (252, 126, 34), (12, 1400, 64), (20, 1344, 40), (16, 960, 70), (8, 1300, 102), (24, 1764, 26),
    (10, 1560, 68)])
def test_plans_against_oracle(orc, cuda, shape):
    """Solve against the oracle (1e-12) and the refined form with two sweeps
    (1e-11, its bar)."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[plans] {shape}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 1.0)
    f = np.random.default_rng(19).standard_normal(g.shape)
    wz = g.dzf[1:-1]
    inner = (slice(1, -1),) * 3
    f[inner] -= (f[inner].sum(axis=(1, 2)) * wz).sum() / (wz.sum() * nx * ny)
    ref = f.copy()
    orc.OraclePPE(nx, ny, nz, g.dx, g.dy, g.dzf, pin_gauge=True).solve(ref)
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    p, q = (torch.from_numpy(f.copy()).to(cuda) for _ in range(2))
    s.solve(p)
    s.solve_refined(q, 2)
    top = np.abs(ref[inner]).max()
    assert np.abs(p.cpu().numpy() - ref)[inner].max() <= 1e-12 * top
    assert np.abs(q.cpu().numpy() - ref)[inner].max() <= 1e-11 * top


# k chunks of odd and even lengths, several and short last ones, with and without
# partial sums of Mean_h
@pytest.mark.parametrize("kc", ["3", "5", "10", "13"])
@pytest.mark.parametrize("forced", [(True, True, False), (False, False, False)])
def test_run_equals_steps_on_chunks(cuda, forced, kc, monkeypatch):
    """pll_channel_run against as many calls of pll_channel_step, bit for bit."""
    import torch
    from powerllel_channel_amd import Channel, PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    monkeypatch.setenv("PLL_RK_KC", kc)
    nx, ny, nz = 70, 26, 29
    print(f"[run = steps] kc={kc} forced={forced}", flush=True)
    g = Grid(nx, ny, nz, 0.1 * nx, 0.1 * ny, 2.0, 2.0)
    ch = Channel(nx, ny, nz, g.lx, g.ly, g.lz, g.dzf, 1e-3, 1e-3, u_crf=0.2, is_forced=forced,
                 vel_force=(1.0, 0.2, 0.0))
    s = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    gen = torch.Generator().manual_seed(8)
    f = [0.3 * torch.randn(g.shape, generator=gen, dtype=torch.float64).to(cuda) for _ in range(3)]
    ch.bc_vel(*f)
    a = [t.clone() for t in f] + [torch.zeros_like(f[0]) for _ in range(4)]
    b = [t.clone() for t in a]
    ch.run(s, 4, *a)
    for _ in range(4):
        ch.step(s, *b)
    for q in (0, 1, 2, 6):
        assert torch.isfinite(b[q]).all()
        assert torch.equal(a[q], b[q]), q


# regular tiles of 4 columns below 5000 columns, ragged ones from there on and
# where there are no regular ones
@pytest.mark.parametrize("shape,rag", [((4, 4, 256), "0"), ((28, 16, 192), "0"),
                                       ((60, 80, 64), "0"), ((60, 84, 64), "1"),
                                       ((100, 100, 128), "1"), ((12, 10, 50), "1")])
def test_fp64_z_tiles_of_4_columns(cuda, shape, rag, monkeypatch):
    """The solve and its transpose are bit for bit those of a solver held to the
    tiles the rule names."""
    import torch
    from powerllel_channel_amd import PoissonSolver
    from powerllel_channel_amd.mesh import Grid
    nx, ny, nz = shape
    print(f"[fp64, 4-column z tiles] {shape}", flush=True)
    g = Grid(nx, ny, nz, 6.0, 3.0, 2.0, 2.0)
    f = torch.from_numpy(np.random.default_rng(23).standard_normal(g.shape)).to(cuda)
    default = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    monkeypatch.setenv("PLL_TRID_RAG", rag)
    held = PoissonSolver(nx, ny, nz, g.dx, g.dy, g.dzf)
    for name in ("solve", "solve_adjoint"):
        p, q = f.clone(), f.clone()
        getattr(default, name)(p)
        getattr(held, name)(q)
        assert torch.isfinite(q).all() and torch.equal(p, q), name
