"""A problem of a batch has the bits of its single solve: whichever variant
the tuner picks (a choice by time) and whatever else is in the batch."""
import pytest

pytestmark = pytest.mark.gpu

FACES = {"dirichlet": (0.0, 1.0, 0.0, 1.0), "robin": (0.5, 1.0, 0.25, 1.5), "periodic": (0.0, 1.0, 0.0, 1.0)}
VARIANTS = (4, 5, 8, 9)  # staged and merged launches, mode-solve tiles of 32 and 64 rows


def problems(specs, form):
    """Plans, right-hand sides, face data and single solves of (nx, ny, N, ne, faces)."""
    import torch
    from mpi_amd.solver import HelmholtzPlan
    gen = torch.Generator(device="cuda").manual_seed(11)
    rand = lambda *s: torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    plans, fs, gs = [], [], []
    for i, (nx, ny, N, ne, faces) in enumerate(specs):
        al, bl, ar, br = FACES[faces]
        p = HelmholtzPlan(nx, ny, N, ne, lam=0.5 + i, alpha_l=al, beta_l=bl, alpha_r=ar, beta_r=br, form=form,
                          periodic_z=faces == "periodic")
        plans.append(p)
        fs.append(rand(nx, ny, p.nz))
        gs.append(None if faces == "periodic" else rand(nx, ny))
    return plans, fs, gs, [p.solve(f, g, g) for p, f, g in zip(plans, fs, gs)]


def same_bits(specs, form, subsets=()):
    """Every variant of the whole batch, and the tuned one of each subset."""
    import torch
    from mpi_amd.solver import BatchSolver
    plans, fs, gs, want = problems(specs, form)
    for picks in [range(len(specs))] + list(subsets):
        pick = lambda v: [v[i] for i in picks]  # noqa: E731
        b = BatchSolver(pick(plans))
        for variant in VARIANTS if len(picks) == len(specs) else (-1,):
            b.force_variant(variant)
            us = b.solve(pick(fs), pick(gs), pick(gs))
            b.status()
            for k, u in zip(picks, us):
                assert torch.equal(u, want[k]), (variant, len(picks), specs[k])
        b.close()
    for p in plans:
        p.close()


def test_mixed_batch(cuda):
    """MIXED problems at every padded size, one element and several, each kind
    of faces."""
    sizes = [(5, 1), (18, 8), (34, 3), (35, 1), (66, 2), (67, 5), (98, 1), (99, 4), (130, 1)]
    same_bits([(nx, ny, N, ne, faces) for (nx, ny) in ((32, 16), (1, 32)) for N, ne in sizes
               for faces in ("dirichlet", "robin", "periodic")]
              + [(64, 64, 67, 10, "periodic"), (64, 64, 98, 4, "robin")], "mixed")


def test_diag_batch_general(cuda):
    """DIAG problems of several elements, Robin faces or periodic z, N - 2 at
    the edges of the column tiles (short elements have a kernel of their own)."""
    sizes = [(3, 1), (5, 16), (9, 8), (18, 16), (19, 3), (34, 8), (35, 1), (66, 2), (67, 1), (99, 4), (130, 1)]
    same_bits([(nx, ny, N, ne, faces) for (nx, ny) in ((32, 16), (1, 32)) for N, ne in sizes
               for faces in ("robin", "periodic", "dirichlet")[:3 if ne > 1 else 2]], "diag")


def test_diag_batch_dirichlet_five_stages(cuda):
    """One-element Dirichlet DIAG problems that stay on the five stages in every
    variant: sides of 16, and so few tiles of larger grids that the z-first
    kernels (whose bits differ) are not taken; every padded size."""
    Ns = (3, 17, 33, 34, 35, 65, 66, 67, 97, 98, 99, 129, 130)
    sides = ((16, 256), (256, 16), (16, 16), (64, 16), (16, 128), (1, 64), (1, 1))
    same_bits([(nx, ny, N, 1, "dirichlet") for nx, ny in sides for N in Ns], "diag")
    same_bits([(32, 32, N, 1, "dirichlet") for N in Ns] + [(32, 64, 130, 1, "dirichlet")], "diag", [[0], [12, 13]])


def test_diag_batch_z_first_bits(cuda):
    """A batch whose one-element Dirichlet problems go z-first: the same bits in
    every variant and in the next solve; those of the single solve where that
    goes z-first too, else equal to rounding (1e-13)."""
    import torch
    from mpi_amd.solver import BatchSolver
    specs = [(nx, ny, N, 1, "dirichlet") for nx, ny in ((32, 32), (32, 256), (64, 64), (128, 64), (128, 128), (256, 32))
             for N in (5, 34, 67, 130)] + [(16, 32, 33, 1, "dirichlet"), (32, 16, 9, 2, "robin")]
    plans, fs, gs, want = problems(specs, "diag")
    b = BatchSolver(plans)
    first = None
    for variant in VARIANTS * 2:
        b.force_variant(variant)
        us = b.solve(fs, gs, gs)
        b.status()
        first = first or [u.clone() for u in us]
        assert all(torch.equal(u, v) for u, v in zip(us, first)), variant
    b.close()
    for spec, p, u, w, f, g in zip(specs, plans, first, want, fs, gs):
        p.profile(True)
        p.solve(f, g, g)
        alone = "xy_filter" in p.profile_read()[0]
        assert torch.equal(u, w) if alone or 16 in spec[:2] else float((u - w).abs().max() / w.abs().max()) <= 1e-13
        p.close()
