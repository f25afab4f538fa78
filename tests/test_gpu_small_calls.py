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
