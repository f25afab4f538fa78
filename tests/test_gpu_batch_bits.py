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
               for faces in ("dirichlet", "robin", "periodic")], "mixed")


def test_diag_batch_general(cuda):
    """DIAG problems of several elements, Robin faces or periodic z, N - 2 at
    the edges of the column tiles (short elements have a kernel of their own)."""
    sizes = [(3, 1), (5, 16), (9, 8), (18, 16), (19, 3), (34, 8), (35, 1), (66, 2), (67, 1), (99, 4), (130, 1)]
    same_bits([(nx, ny, N, ne, faces) for (nx, ny) in ((32, 16), (1, 32)) for N, ne in sizes
               for faces in ("robin", "periodic", "dirichlet")[:3 if ne > 1 else 2]], "diag")
