"""Small problems and many of them: the kernels that hold these sizes, against
the others bit for bit or against the oracle, and how long the calls take
relative to one another (where a kernel for larger sizes took several times as
long)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def best_us(fn, reps=20, rounds=7):
    """Least mean time of `reps` calls over `rounds`, microseconds."""
    import torch
    fn()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(rounds):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(reps):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / reps)
    return best


def factored(n, count, seed):
    import torch
    from mpi_amd.solver import lu_factor_batched
    gen = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn((count, n, n), dtype=torch.float64, device="cuda", generator=gen)
    b = torch.randn((count, n), dtype=torch.float64, device="cuda", generator=gen)
    piv, _, _ = lu_factor_batched(A)
    return A, piv, b


@pytest.mark.parametrize("n", [1, 2, 3])
def test_lu_solve_of_many_tiny_systems_is_bound_by_memory(cuda, n):
    """524,288 systems: the matrices, pivots and vectors at half a TB/s (a
    sixteenth of the card's rate) and a launch."""
    from mpi_amd.solver import lu_solve_batched
    count = 524288
    A, piv, b = factored(n, count, n)
    took = best_us(lambda: lu_solve_batched(A, piv, b))
    assert took <= 10 + count * (8 * n * n + 4 * (n - 1) + 16 * n) / 0.5e6


@pytest.mark.parametrize("n", [1, 4, 6, 7, 8, 10, 11])
def test_lu_solve_same_bits_however_many(cuda, n):
    """A system's result does not depend on how many there are (one thread or
    one wave per system)."""
    import torch
    from mpi_amd.solver import lu_solve_batched
    A, piv, b = factored(n, 20000, 40 + n)
    x = lu_solve_batched(A, piv, b.clone())
    for lo, hi in ((0, 7), (19000, 20000)):
        y = lu_solve_batched(A[lo:hi].clone(), piv[lo:hi].clone(), b[lo:hi].clone())
        assert torch.equal(x[lo:hi], y)


def test_lu_solve_of_more_systems_than_one_launch_holds(cuda):
    """2^26 + 70 systems of 7 (a wave each: more than 2^32 threads): every one is solved."""
    import torch
    from mpi_amd.solver import lu_solve_batched
    n, count = 7, (1 << 26) + 70
    A, piv, b = factored(n, 1000, 3)
    want = lu_solve_batched(A, piv, b.clone())
    reps = -(-count // 1000)
    x = b.repeat(reps, 1)[:count].contiguous()
    LU, pv = A.repeat(reps, 1, 1)[:count].contiguous(), piv.repeat(reps, 1)[:count].contiguous()
    lu_solve_batched(LU, pv, x)
    assert torch.equal(x[:count // 1000 * 1000].view(-1, 1000, n),
                       want.expand(count // 1000, 1000, n)) and torch.equal(x[-(count % 1000):], want[:count % 1000])


@pytest.mark.parametrize("N", [129, 257])
def test_derivative_z_of_few_columns_is_short(cuda, N):
    """One column (a 1-D problem's field) is spread over the chip: at most 0.6 of
    the time of 16,384 columns, one tile per CU."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    took = []
    for side in (1, 128):
        plan = HelmholtzPlan(side, side, N, 1, form="diag")
        u = torch.randn((1, side, side, N), dtype=torch.float64, device="cuda")
        out = torch.empty_like(u)
        took.append(best_us(lambda: plan.derivative_z(u, 1, out=out)))
        plan.close()
    assert took[0] <= 0.6 * took[1], took


@pytest.mark.parametrize("nx,ny,N", [(1, 1, 3), (1, 1, 258), (16, 64, 256), (32, 32, 257), (64, 64, 64), (64, 64, 65),
                                     (128, 128, 16), (128, 128, 17)])
def test_derivative_z_few_and_many_outputs(cuda, nx, ny, N):
    """One thread per output (to 2^18 outputs), tiles of 64 columns above and
    where the output is the input: the reference's products and sums in its
    order, bit for bit."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    plan = HelmholtzPlan(nx, ny, N, 1, form="diag")
    gen = torch.Generator(device="cuda").manual_seed(N)
    u = torch.randn((1, nx, ny, N), dtype=torch.float64, device="cuda", generator=gen)
    for order, D in zip((1, 2), plan.operators()):
        Dd = torch.from_numpy(np.ascontiguousarray(D)).cuda()
        want = torch.zeros_like(u)
        for p in range(N):  # p ascending, every product rounded before it is added
            want = want + Dd[:, p] * u[..., p:p + 1]
        assert torch.equal(plan.derivative_z(u, order, out=torch.empty_like(u)), want)
        same = u.clone()
        plan.derivative_z(same, order, out=same)
        assert torch.equal(same, want)
    plan.close()


@pytest.mark.parametrize("N", [3, 4])
def test_plain_smallest_operators_are_short(cuda, N):
    """The reference algorithm with one or two interior nodes against seven: at
    most four fifths of the time (16-column panels cost nearly the same)."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    took = []
    for n in (N, 9):
        plan = HelmholtzPlan(128, 128, n, 1, lam=3.0, form="plain")
        f = torch.randn((128, 128, n), dtype=torch.float64, device="cuda")
        g = torch.randn((128, 128), dtype=torch.float64, device="cuda")
        u = plan.empty_field()
        took.append(best_us(lambda: plan.solve(f, g, g, out=u)))
        plan.close()
    assert took[0] <= 0.8 * took[1], took


@pytest.mark.parametrize("nx,ny,N,ne", [(1, 1, 3, 1), (256, 64, 3, 4), (128, 128, 4, 1), (128, 128, 4, 2),
                                        (128, 256, 5, 1), (256, 256, 5, 1), (128, 128, 6, 1), (256, 128, 6, 1),
                                        (64, 64, 7, 1), (128, 64, 7, 1), (1, 64, 8, 12), (1, 64, 8, 13),
                                        (64, 32, 10, 1), (64, 64, 10, 1), (32, 32, 12, 1), (64, 32, 12, 1),
                                        (16, 16, 14, 1), (32, 32, 14, 1), (1, 64, 16, 1), (1, 128, 16, 2),
                                        (32, 32, 20, 1), (64, 32, 20, 1), (16, 16, 24, 1), (1, 64, 35, 1),
                                        (1, 64, 37, 1), (16, 16, 37, 1)])
def test_plain_both_kernels_at_the_line_between_them(cuda, nx, ny, N, ne):
    """Sizes on either side of the rule that sends small operators of few modes
    to the stepwise kernel: against the oracle within twice its rounding spread
    (or 1e-12), every instance with the same bits."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    from oracle import pyoracle as po
    lam = 3.0
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    plan = HelmholtzPlan(nx, ny, N, ne, lam=lam, form="plain", **geo)
    r = np.random.default_rng(N + ne)
    f = r.standard_normal((nx, ny, plan.nz))
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    dev = [torch.from_numpy(v).cuda() for v in (f, *g)]
    desc = po.make_desc(nx, ny, ne * N, N, size=1, lam=lam, **geo)
    uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    u = plan.solve(*dev)
    plan.status()
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    for cols in plan.diag_candidates():
        plan.set_diag_tile(cols)
        assert torch.equal(plan.solve(*dev), u)
        plan.status()
    plan.close()


@pytest.mark.parametrize("N", [7, 9, 11, 16, 19, 24, 35])
@pytest.mark.parametrize("scale", ["unit", "rows", "small", "huge"])
def test_plain_panels_of_small_operators_on_many_modes(cuda, N, scale):
    """The panel kernel's first columns and a second panel of few, on operators
    of their own for every mode that exchange rows at almost every step (rows of
    very different scale; scales whose reciprocals leave the ordinary range): u
    per mode from numpy's solve.  Elimination with partial pivoting: n eps times
    the condition, and a growth of 8; a mode with a zero column is singular."""
    import torch
    from mpi_amd._lib import HzError
    from mpi_amd.solver import HelmholtzPlan
    nx, ny, n = 128, 64, N - 2
    plan = HelmholtzPlan(nx, ny, N, 1, form="plain")
    M = ny // 2 + 1
    r = np.random.default_rng(N)
    A = r.standard_normal((nx // 2 + 1, M, n, n)) + 2.0 * np.eye(n)
    s = {"unit": np.ones(n), "rows": 10.0 ** r.integers(-6, 7, n), "small": np.full(n, 2.0 ** -600),
         "huge": np.full(n, 2.0 ** 1000)}[scale]
    w = {"unit": 1.0, "rows": 1.0, "small": 2.0 ** -600, "huge": 2.0 ** 900}[scale]  # of the right-hand side
    f = r.standard_normal((nx, ny, N)) * w
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    zero = dev(np.zeros((nx, ny)))
    op = (s[:, None] * A).reshape(-1, n, n)
    u = plan.solve_operators(dev(f), zero, zero, op_full=dev(op)).cpu().numpy()
    plan.status()
    F = np.fft.rfft2(f[:, :, 1:-1] / w, axes=(0, 1))
    ix = np.minimum(np.arange(nx), nx - np.arange(nx))
    As = A[ix]                                              # [nx, M, n, n]
    ratio = s / w
    W = np.linalg.solve(As, (F / ratio)[..., None])[..., 0]
    want = np.fft.irfft2(W, s=(nx, ny), axes=(0, 1))
    # a mode's error, n eps cond |u|, and its sum over the modes in the transform back
    tol = 8 * n * 2.0 ** -52 * (np.linalg.cond(As) * np.abs(W).max(-1)).sum() * 2 / (nx * ny)
    assert np.abs(u[:, :, 1:-1] - want).max() <= tol
    op[7, :, n // 2] = 0.0
    plan.solve_operators(dev(f), zero, zero, op_full=dev(op))
    with pytest.raises(HzError):
        plan.status()
    plan.close()


@pytest.mark.parametrize("nx,ny,N,ne,periodic", [(32, 32, 67, 9, True), (32, 32, 98, 8, True), (64, 64, 67, 4, False),
                                                 (64, 64, 98, 3, False), (32, 32, 66, 8, False)])
def test_mixed_both_kernels_at_the_line_between_them(cuda, nx, ny, N, ne, periodic):
    """MIXED solves on either side of the rule that sends several elements of 67
    to 98 points to the four-wave tile: against the oracle within twice its
    rounding spread (or 1e-12), the residual history falling."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    from oracle import pyoracle as po
    lam = 3.0
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    plan = HelmholtzPlan(nx, ny, N, ne, lam=lam, form="mixed", periodic_z=periodic, **geo)
    r = np.random.default_rng(N + ne)
    f = r.standard_normal((nx, ny, plan.nz))
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    dev = lambda v: torch.from_numpy(v).cuda()  # noqa: E731
    desc = po.make_desc(nx, ny, ne * N, N, size=1, lam=lam, **geo)
    if periodic:
        f[:, :, -1] = f[:, :, 0]
        uo, uf = po.solve_periodic(desc, f), po.solve_periodic(desc, f, fma=True)
        u = plan.solve(dev(f))
    else:
        uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
        u = plan.solve(dev(f), *map(dev, g))
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    h = plan.mixed_history()
    assert len(h) == 2 and 0 < h[1] < h[0] < 1e-3
    plan.close()
