"""The z-first solve at the sizes where its eigenvector correction is largest."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [122, 123, 124, 125, 126, 127, 128])
def test_z_first_solve_where_the_correction_is_largest(cuda, N):
    """Nearly equal even/odd eigenvalue pairs (G to 3e-6 in its FP64 block, to
    4.5e-11 in bf16): alone and in a batch, against the oracle within twice its
    rounding spread (or 1e-12)."""
    import torch
    from mpi_amd.solver import BatchSolver, HelmholtzPlan
    nx, ny, lam = 128, 64, 1e-3
    geo = dict(xl=0, xr=2.0, yl=0, yr=3.0, zl=0, zr=2)
    plan = HelmholtzPlan(nx, ny, N, 1, lam=lam, form="diag", **geo)
    r = np.random.default_rng(N)
    f, gl, gr = r.standard_normal((nx, ny, N)), r.standard_normal((nx, ny)), r.standard_normal((nx, ny))
    dev = [torch.from_numpy(v).cuda() for v in (f, gl, gr)]
    desc = po.make_desc(nx, ny, N, N, size=1, lam=lam, **geo)
    uo, uf = po.solve(desc, f, gl, gr), po.solve(desc, f, gl, gr, fma=True)
    bar = max(1e-12, 2.0 * np.abs(uf - uo).max() / np.abs(uo).max())
    plan.profile(True)
    u = plan.solve(*dev)
    assert "xy_filter" in plan.profile_read()[0]
    plan.profile(False)
    assert np.abs(u.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    b = BatchSolver([plan])
    v = b.solve([dev[0]], [dev[1]], [dev[2]])[0]
    b.status()
    assert np.abs(v.cpu().numpy() - uo).max() <= bar * np.abs(uo).max()
    b.close()
    plan.close()
