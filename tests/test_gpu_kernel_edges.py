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
