"""Kernel variants at the sizes where they can go wrong (tile edges,
remainders, the smallest and largest of their range) against the oracle."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def to_dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def factored(n, count, seed, swaps=True):
    """Reference factors and pivots of random systems (rows exchanged at
    almost every step without `swaps` = False's dominant diagonal)."""
    r = np.random.default_rng(seed)
    A = r.standard_normal((count, n, n))
    if not swaps:
        A += 3 * n * np.eye(n)
    b = r.standard_normal((count, n))
    LU, piv, x = np.empty_like(A), np.zeros((count, max(n - 1, 1)), np.int32), np.empty_like(b)
    for c in range(count):
        lu, p, _ = po.lu(A[c])
        LU[c], piv[c, :n - 1] = lu, p
        x[c] = po.lu_solve(lu, p, b[c])
    return LU, piv, b, x


@pytest.mark.parametrize("n", [2, 3, 8, 9, 16, 17, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("swaps", [True, False])
def test_lu_solve_every_size_class(cuda, n, swaps):
    """One wave per system (one row per lane to 64, two to 128), and the
    general kernel above: the reference's result bit for bit."""
    from mpi_amd.solver import lu_solve_batched
    LU, piv, b, x = factored(n, 5, n, swaps)
    got = lu_solve_batched(to_dev(LU), to_dev(piv), to_dev(b)).cpu().numpy()
    assert np.array_equal(got, x)


@pytest.mark.parametrize("nx,ny,N,ne", [(1, 1, 3, 1), (2, 1, 16, 1), (1, 64, 17, 1), (8, 8, 32, 2), (4, 32, 33, 3),
                                        (2, 64, 129, 1), (1, 128, 130, 1), (2, 32, 257, 1), (1, 16, 258, 1)])
def test_derivative_z_tiles(cuda, nx, ny, N, ne):
    """Whole and partial tiles of 64 columns, odd and even column strides,
    one to 17 strips of 16 output rows, both orders: the products and sums of
    the reference in its order, bit for bit."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    plan = HelmholtzPlan(nx, ny, N, ne, form="diag")
    u = np.random.default_rng(N).standard_normal((ne, nx, ny, N))
    du = to_dev(u)
    for order, D in zip((1, 2), plan.operators()):
        want = np.zeros_like(u)
        for p in range(N):  # p ascending, every product rounded before it is added
            want = want + D[:, p] * u[..., p:p + 1]
        got = plan.derivative_z(du, order, out=torch.empty_like(du)).cpu().numpy()
        assert np.array_equal(got, want), order


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("swaps", [True, False])
def test_lu_factor_every_size_class(cuda, n, swaps):
    """One wave per matrix (16, 32, 64 columns) and the work-group kernel
    above: factors, pivots and determinant of the reference bit for bit, and a
    singular matrix flagged."""
    from mpi_amd.solver import lu_factor_batched
    r = np.random.default_rng(n)
    A = r.standard_normal((4, n, n)) + (0 if swaps else 3 * n * np.eye(n))
    A[3] *= 1e-2 ** r.integers(0, 6, (n, 1))  # rows of very different scale
    dA = to_dev(A)
    piv, det, st = (t.cpu().numpy() for t in lu_factor_batched(dA))
    LU = dA.cpu().numpy()
    for c in range(4):
        lu, p, d = po.lu(A[c])
        assert np.array_equal(LU[c], lu) and list(piv[c, :n - 1]) == list(p[:n - 1]) and det[c] == d, c
    assert not st.any()
    if n > 1:
        A[2, :, n // 2 if n > 2 else 0] = 0.0
        st = lu_factor_batched(to_dev(A))[2].cpu().numpy()
        assert list(st) == [0, 0, 4, 0]


@pytest.mark.parametrize("N", [3, 9, 16, 17, 18, 19, 33, 34, 35, 50, 51, 65, 66])
@pytest.mark.parametrize("scale", ["unit", "rows", "small", "huge"])
def test_plain_panel_kernel_any_operator(cuda, N, scale):
    """The mode kernel for N - 2 <= 64 (panels of 16 columns on 16 x 16
    tiles) at its tile edges, on operators that exchange rows at almost every
    step: rows of very different scale, pivots far from 1, and scales whose
    reciprocals leave the ordinary range (the exact pivot comparison).  One
    mode (1-D), Dirichlet ends: A u = f - Dzz[:,0] g_l - Dzz[:,-1] g_r."""
    from mpi_amd.solver import HelmholtzPlan
    n = N - 2
    plan = HelmholtzPlan(1, 1, N, 1, form="plain")
    r = np.random.default_rng(N)
    A = r.standard_normal((n, n)) + (2.0 if n == 1 else 0.0)
    s = {"unit": np.ones(n), "rows": 10.0 ** r.integers(-6, 7, n), "small": np.full(n, 2.0 ** -600),
         "huge": np.full(n, 2.0 ** 1003)}[scale]
    f = r.standard_normal(N)
    b = f.copy()
    b[1:-1] *= s
    zero = to_dev(np.zeros((1, 1)))
    u = plan.solve_operators(to_dev(b.reshape(1, 1, N)), zero, zero, op_full=to_dev((s[:, None] * A)[None]))
    plan.status()
    u = u.cpu().numpy().ravel()
    want = np.linalg.solve(A, f[1:-1])
    # backward stable elimination: n eps times the condition, and a growth of 8
    tol = 8 * n * 2.0 ** -52 * np.linalg.cond(A) * np.abs(want).max()
    assert u[0] == 0 and u[-1] == 0
    assert np.abs(u[1:-1] - want).max() <= tol, (np.abs(u[1:-1] - want).max(), tol)
    if n > 1:  # a zero column is singular
        A[:, n // 2] = 0.0
        plan.solve_operators(to_dev(b.reshape(1, 1, N)), zero, zero, op_full=to_dev((s[:, None] * A)[None]))
        from mpi_amd._lib import HzError
        with pytest.raises(HzError):
            plan.status()
    plan.close()


@pytest.mark.parametrize("nx,ny,N,ne,periodic", [(1, 1, 8, 127, False), (4, 4, 10, 63, False), (4, 2, 66, 7, False),
                                                 (2, 4, 66, 40, True), (4, 4, 18, 16, True), (4, 4, 34, 21, False)])
def test_plain_panel_kernel_many_right_hand_sides(cuda, nx, ny, N, ne, periodic):
    """Up to the largest number of right-hand sides (2 + c ne, c = 2 or 4), in
    one and several groups of 64, against the diagonalised or the reference's
    algorithm (the oracle), within twice the oracle's rounding spread."""
    from mpi_amd.solver import HelmholtzPlan
    lam = 3.0
    plan = HelmholtzPlan(nx, ny, N, ne, xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2, lam=lam, form="plain",
                         periodic_z=periodic)
    r = np.random.default_rng(N + ne)
    f = r.standard_normal((nx, ny, plan.nz))
    if periodic:
        f[:, :, -1] = f[:, :, 0]
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    desc = po.make_desc(nx, ny, ne * N, N, size=1, xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2, lam=lam)
    if periodic:
        uo, uf = po.solve_periodic(desc, f), po.solve_periodic(desc, f, fma=True)
        u = plan.solve(to_dev(f))
    else:
        uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
        u = plan.solve(to_dev(f), *map(to_dev, g))
    plan.status()
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    assert np.abs(u.cpu().numpy() - uo).max() / np.abs(uo).max() <= bar
    plan.close()


@pytest.mark.parametrize("nx,ny,N", [(64, 128, 66), (128, 64, 67), (256, 32, 98), (64, 256, 3), (128, 128, 4),
                                     (256, 64, 17), (64, 256, 18), (128, 256, 19), (256, 128, 34), (256, 256, 5),
                                     (128, 128, 35), (256, 64, 66), (64, 128, 99), (128, 64, 129), (256, 32, 130)])
def test_z_first_solve_every_grid(cuda, nx, ny, N):
    """The one-element Dirichlet DIAG solve with the z contractions outside
    the transforms: every grid it holds, N - 2 at the edges of the matrix
    tiles, end values scaled by beta.  Solve against the oracle within twice
    its rounding spread (or 1e-12); right-hand side a3 u^3 + a1 u bit for bit
    the solve of that field; adjoint (and solve) against the general path,
    which a vanishing Robin term selects, each side within that bar."""
    import torch
    from mpi_amd import _lib
    from mpi_amd.solver import HelmholtzPlan
    lam, bl, br = 3.0, 2.0, -0.5
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    plan = HelmholtzPlan(nx, ny, N, 1, lam=1.0, beta_l=bl, beta_r=br, form="diag", **geo)
    plan.set_lambda(lam)
    r = np.random.default_rng(nx + ny + N)
    f = r.standard_normal((nx, ny, N))
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    df, dg = to_dev(f), [to_dev(v) for v in g]
    desc = po.make_desc(nx, ny, N, N, size=1, lam=lam, betal=bl, betar=br, **geo)
    uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    plan.profile(True)
    u = plan.solve(df, *dg)
    assert "xy_filter" in plan.profile_read()[0]
    plan.profile(False)
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    lib = _lib.load()
    cub = torch.empty_like(df)
    _lib.check(lib.hz_cubic_rhs(df.data_ptr(), cub.data_ptr(), df.numel(), 0.5, -2.0,
                                torch.cuda.current_stream().cuda_stream))
    assert torch.equal(plan.solve_cubic(df, 0.5, -2.0, *dg), plan.solve(cub, *dg))
    other = HelmholtzPlan(nx, ny, N, 1, lam=lam, alpha_l=1e-300, beta_l=bl, alpha_r=1e-300, beta_r=br, form="diag",
                          **geo)
    pairs = [(u, other.solve(df, *dg))] + list(zip(plan.adjoint(df)[:3], other.adjoint(df)[:3]))
    for got, want in pairs:
        assert float((got - want).abs().max()) <= 2 * bar * float(want.abs().max())
    plan.close()
    other.close()


@pytest.mark.parametrize("nx,ny,lanes", [(32, 32, 1), (64, 32, 7), (32, 64, 65), (128, 32, 33), (64, 128, 31),
                                         (256, 64, 17), (32, 256, 15), (256, 128, 9), (16, 512, 3)])
@pytest.mark.parametrize("order", [1, 2])
def test_fourier_derivative_lines(cuda, nx, ny, lanes, order):
    """The one-pass Fourier derivative at every line length it holds (and one
    axis below and above them), whole and partial lane tiles, in place, and
    onto an output that overlaps the input, against numpy's transform in 64
    bits.  Two transforms of log2 L levels, at most four roundings each on
    values whose largest is about the result's: 16 log2 L 2^-53 of it."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    lx, ly = 3.0, 2.0
    plan = HelmholtzPlan(nx, ny, 3, 1, xl=0, xr=lx, yl=0, yr=ly, form="diag")
    u = np.random.default_rng(nx + ny + lanes).standard_normal((nx, ny, lanes))
    du = to_dev(u)
    for axis, L, length in ((0, nx, lx), (1, ny, ly)):
        k = np.fft.fftfreq(L, 1.0 / L).reshape((-1, 1, 1) if axis == 0 else (1, -1, 1))
        want = np.fft.ifft(np.fft.fft(u, axis=axis) * (2j * np.pi * k / length) ** order, axis=axis).real
        tol = 16 * np.log2(L) * 2.0 ** -53 * np.abs(want).max()
        got = plan.derivative_xy(du, axis, order)
        assert np.abs(got.cpu().numpy() - want).max() <= tol
        same = du.clone()
        plan.derivative_xy(same, axis, order, out=same)
        assert torch.equal(same, got)
        buf = torch.empty(u.size + 5, dtype=torch.float64, device="cuda")
        src, dst = buf[:u.size].view(u.shape), buf[5:].view(u.shape)
        src.copy_(du)
        plan.derivative_xy(src, axis, order, out=dst)
        assert np.abs(dst.cpu().numpy() - want).max() <= tol
    plan.close()


@pytest.mark.parametrize("N", [3, 4, 17, 18, 19, 34, 35, 66, 67, 98, 99, 130])
@pytest.mark.parametrize("faces,ne", [("dirichlet", 1), ("robin", 1), ("robin", 3), ("periodic", 1), ("periodic", 8)])
def test_mixed_one_wave_per_16_columns(cuda, N, faces, ne):
    """The MIXED mode solve for N - 2 <= 128 at the edges of its column tiles,
    with whole and partial row tiles, against the oracle within twice its
    rounding spread (or 1e-12), and its residual history present and falling."""
    from mpi_amd.solver import HelmholtzPlan
    nx, ny, lam = 4, 8, 3.0
    ab = (0.7, 1.3, 0.4, 2.0) if faces == "robin" else (0.0, 2.0, 0.0, -0.5)
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    kw = {} if faces == "periodic" else dict(alpha_l=ab[0], beta_l=ab[1], alpha_r=ab[2], beta_r=ab[3])
    plan = HelmholtzPlan(nx, ny, N, ne, lam=lam, form="mixed", periodic_z=faces == "periodic", **geo, **kw)
    r = np.random.default_rng(N + ne)
    f = r.standard_normal((nx, ny, plan.nz))
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    dk = {} if faces == "periodic" else dict(alphal=ab[0], betal=ab[1], alphar=ab[2], betar=ab[3])
    desc = po.make_desc(nx, ny, ne * N, N, size=1, lam=lam, **geo, **dk)
    if faces == "periodic":
        f[:, :, -1] = f[:, :, 0]
        uo, uf = po.solve_periodic(desc, f), po.solve_periodic(desc, f, fma=True)
        u = plan.solve(to_dev(f))
    else:
        uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
        u = plan.solve(to_dev(f), *map(to_dev, g))
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    h = plan.mixed_history()
    assert len(h) == 2 and 0 < h[1] < h[0] < 1e-3
    plan.close()


@pytest.mark.parametrize("N,ne", [(3, 1), (4, 64), (9, 5), (17, 13), (18, 1), (18, 63), (19, 1), (19, 32), (33, 3),
                                  (34, 7), (34, 31)])
@pytest.mark.parametrize("faces", ["robin", "periodic", "dirichlet"])
def test_diag_short_elements(cuda, N, ne, faces):
    """The DIAG mode solve of several elements, Robin faces or periodic z at
    N - 2 <= 32: 16 and 32 columns, whole and partial row tiles, up to the
    largest element count of a tile.  Solve against the oracle within twice
    its rounding spread (or 1e-12); adjoint by <S x, v> = <x, S^T v>."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    nx, ny, lam = 4, 8, 3.0
    ab = (0.7, 1.3, 0.4, 2.0) if faces == "robin" else (0.0, 2.0, 0.0, -0.5)
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    per = faces == "periodic"
    kw = {} if per else dict(alpha_l=ab[0], beta_l=ab[1], alpha_r=ab[2], beta_r=ab[3])
    plan = HelmholtzPlan(nx, ny, N, ne, lam=lam, form="diag", periodic_z=per, **geo, **kw)
    r = np.random.default_rng(N + ne)
    f = r.standard_normal((nx, ny, plan.nz))
    g = [r.standard_normal((nx, ny)) for _ in range(2)]
    dk = {} if per else dict(alphal=ab[0], betal=ab[1], alphar=ab[2], betar=ab[3])
    desc = po.make_desc(nx, ny, ne * N, N, size=1, lam=lam, **geo, **dk)
    df, dg = to_dev(f), [] if per else [to_dev(v) for v in g]
    if per:
        f[:, :, -1] = f[:, :, 0]
        df = to_dev(f)
        uo, uf = po.solve_periodic(desc, f), po.solve_periodic(desc, f, fma=True)
    else:
        uo, uf = po.solve(desc, f, *g), po.solve(desc, f, *g, fma=True)
    u = plan.solve(df, *dg)
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    v = to_dev(r.standard_normal(u.shape))
    fbar, glbar, grbar, _ = plan.adjoint(v)
    lhs = float((u * v).sum())
    rhs = float((df * fbar).sum()) + (0.0 if per else float((dg[0] * glbar).sum() + (dg[1] * grbar).sum()))
    scale = float((df * fbar).abs().sum() + (u * v).abs().sum())
    assert abs(lhs - rhs) <= bar * scale
    plan.close()


def test_batch_z_first_every_grid(cuda):
    """The z-first part of a batch: every grid it holds beside one that it
    does not, N - 2 at the edges of the matrix tiles (partial groups of tiles
    included), then with one plan's lambda changed and one turned to Robin
    faces (which leaves this path), against the oracle within twice its
    rounding spread (or 1e-12)."""
    from mpi_amd.solver import BatchSolver, HelmholtzPlan
    sides, Ns = (32, 64, 128, 256), (130, 99, 67, 35, 98, 66, 34, 19, 33, 17, 9, 6, 18, 5, 4, 3)
    specs = sorted(((nx, ny) for nx in sides for ny in sides), key=lambda s: s[0] * s[1])
    specs = [(nx, ny, N) for (nx, ny), N in zip(specs, Ns)] + [(16, 64, 34), (32, 32, 3)]
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    lam = [0.5 + i for i in range(len(specs))]
    robin = [(0.0, 2.0, 0.0, -0.5)] * len(specs)
    plans = [HelmholtzPlan(nx, ny, N, 1, lam=l, beta_l=2.0, beta_r=-0.5, form="diag", **geo)
             for (nx, ny, N), l in zip(specs, lam)]
    r = np.random.default_rng(7)
    f = [r.standard_normal(s) for s in specs]
    g = [[r.standard_normal(s[:2]) for s in specs] for _ in range(2)]
    batch = BatchSolver(plans)
    for rep in range(2):
        us = batch.solve([to_dev(v) for v in f], [to_dev(v) for v in g[0]], [to_dev(v) for v in g[1]])
        batch.status()
        for k, (nx, ny, N) in enumerate(specs):
            if rep and k not in (3, 5, 6):
                continue
            al, bl, ar, br = robin[k]
            desc = po.make_desc(nx, ny, N, N, size=1, lam=lam[k], alphal=al, betal=bl, alphar=ar, betar=br, **geo)
            uo, uf = (po.solve(desc, f[k], g[0][k], g[1][k], fma=m) for m in (False, True))
            bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
            assert np.abs(us[k].cpu().numpy() - uo).max() <= bar * np.abs(uo).max(), (rep, specs[k])
        lam[3], robin[5] = 40.0, (0.7, 1.3, 0.4, 2.0)
        plans[3].set_lambda(lam[3])
        plans[5].set_robin(*robin[5])
    batch.close()
    for p in plans:
        p.close()
