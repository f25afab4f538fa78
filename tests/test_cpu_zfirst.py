"""The z-first solve's eigenvector correction G is small enough for the
precisions it is applied in, at every size that the kernels take."""
import ctypes
import os
import re

import numpy as np
import pytest

PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mpi_amd", "csrc", "plan.cpp")


def correction(N, lz):
    """|G| of the even/odd eigenbasis, G_ij = M_ij / (mu_j - mu_i) between the
    halves, M = Winv F Ea F^-1 W with Ea the antisymmetric part of the interior
    operator: its maximum in the first 16 of each half and elsewhere."""
    from mpi_amd import _lib
    lib = _lib.load()
    ptr = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))  # noqa: E731
    m = N - 2
    NP = max(32, -(-m // 32) * 32)
    H, ho = NP // 2, m // 2
    he = m - ho
    mu, W, Wi, D = np.zeros(NP), np.zeros((NP, NP)), np.zeros((NP, NP)), np.zeros((N, N))
    _lib.check(lib.hz_host_eigen_split(N, 1, lz, NP, ptr(mu), ptr(W), ptr(Wi), None))
    _lib.check(lib.hz_host_plan_operators(N, 1, lz, None, None, None, ptr(D)))
    A = D[1:-1, 1:-1].astype(np.longdouble)
    F, Fi = np.zeros((NP, m), np.longdouble), np.zeros((m, NP), np.longdouble)
    for i in range(ho):
        F[i, i] = F[i, m - 1 - i] = F[H + i, i] = 1
        F[H + i, m - 1 - i] = -1
        Fi[i, i] = Fi[m - 1 - i, i] = Fi[i, H + i] = 0.5
        Fi[m - 1 - i, H + i] = -0.5
    if m % 2:
        F[ho, ho] = Fi[ho, ho] = 1
    M = Wi.astype(np.longdouble) @ (F @ ((A - A[::-1, ::-1]) / 2 @ (Fi @ W.astype(np.longdouble))))
    r = np.r_[0:he, H:H + ho]
    cross = (r >= H)[:, None] != (r >= H)[None, :]
    gap = np.where(cross, mu[r][None, :] - mu[r][:, None], 1)
    G = np.abs(np.where(cross, M[np.ix_(r, r)] / gap, 0)).astype(float)
    block = (r % H < 16)[:, None] & (r % H < 16)[None, :]
    return G[block].max(initial=0), G[~block].max(initial=0)


@pytest.mark.parametrize("lz", [2.0, 3.7])
def test_z_first_correction_is_within_its_bounds(lz):
    """At every N from 3 to 130, with room to spare: the plan gives the z-first
    operands up only above these bounds."""
    text = open(PLAN).read()
    block, rest = map(float, re.search(r"kZfBlock = ([\d.e-]+), kZfRest = ([\d.e-]+);", text).groups())
    for N in range(3, 131):
        in_block, elsewhere = correction(N, lz)
        assert in_block <= block / 2 and elsewhere <= rest / 2, (N, in_block, elsewhere)
