"""Runs of one and two steps: the many-step kernel takes those on plates with
four stages a step, whose passes it saves, and leaves the others, which are a
launch or two of the streaming kernels, where they were; from three steps on it
takes all (no GPU needed)."""

import ctypes

import pytest

from pararealml_amd import _native as nat


def _steps(eq, integ, prec, ndim, n, n_steps, n_grids=1):
    grids = (nat.PmlGrid * n_grids)()
    for g in grids:
        g.n0, g.n1, g.dx0, g.dx1 = (n if ndim == 2 else 1), n, 0.1, 0.1
    plan = (ctypes.c_int * 4)()
    nat.check(nat.load_library().pml_fdm_auto_plan(nat.PML_EQ[eq], integ, prec, ndim, grids,
                                                   n_grids, n_steps, plan))
    return plan[3]


@pytest.mark.parametrize("prec", [nat.PML_F64, nat.PML_F32, nat.PML_F32C])
@pytest.mark.parametrize("n,n_grids", [(33, 1), (33, 64), (257, 1), (600, 1)])
@pytest.mark.parametrize("eq", ["diffusion", "convection_diffusion", "wave", "burgers",
                                "shallow_water", "cahn_hilliard"])
def test_short_runs(eq, n, n_grids, prec):
    for integ in (nat.PML_INT_FE, nat.PML_INT_MIDPOINT, nat.PML_INT_RK4):
        # a stage is a step where the right-hand side does not see it
        staged = integ == nat.PML_INT_RK4 and eq != "cahn_hilliard"
        for n_steps in (1, 2):
            assert (_steps(eq, integ, prec, 2, n, n_steps, n_grids) > 0) == staged
        assert _steps(eq, integ, prec, 2, n, 3, n_grids) > 0


def test_short_runs_on_lines():
    for eq in ("burgers", "diffusion", "wave"):
        for integ in (nat.PML_INT_FE, nat.PML_INT_RK4):
            for n_steps in (1, 2):
                assert _steps(eq, integ, nat.PML_F64, 1, 500, n_steps) == 0
            assert _steps(eq, integ, nat.PML_F64, 1, 500, 3) == 3
