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
