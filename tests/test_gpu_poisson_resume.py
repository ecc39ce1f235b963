"""A Poisson time loop one of whose solves needs more sweeps than the loop on
the device takes: the run goes on from the last steps that were whole, with
the same states, instead of from its start."""

import numpy as np
import pytest

import pararealml_amd as pml
from tests.helpers import navier_stokes_cavity

pytestmark = pytest.mark.gpu


class _Library:
    """The library, with the device loop reported as unfinished from its
    step `fails_at` on, and the single steps counted."""

    def __init__(self, lib, fails_at):
        self._lib, self._fails_at = lib, fails_at
        self.steps = self.single = 0

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def pml_fdm_poisson_solve(self, *args):
        rc = self._lib.pml_fdm_poisson_solve(*args)
        self.steps += args[11]
        if self.steps > self._fails_at:
            args[-2]._obj.value = 0
        return rc

    def pml_fdm_solve(self, *args):
        self.single += args[15]
        return self._lib.pml_fdm_solve(*args)


# (steps, snapshots every, the first step that fails, steps taken one by one)
RUNS = [(12, 1, 99, 0), (12, 1, 6, 8), (12, 2, 9, 4), (12, 3, 2, 12), (12, 6, 9, 6),
        (12, 12, 3, 12), (12, 12, 11, 4), (10, 1, 9, 2)]


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("steps,every,fails_at,single", RUNS)
def test_runs_resume_from_their_last_whole_steps(steps, every, fails_at, single, precision,
                                                 monkeypatch):
    from pararealml_amd import _native as nat
    from pararealml_amd.operators.fdm import (
        RK4, FDMOperator, ThreePointCentralDifferenceMethod, fdm_operator)

    print(f"case: poisson resume {steps}/{every} {fails_at} {precision}", flush=True)
    monkeypatch.setattr(fdm_operator, "_POISSON_STEPS", 4, raising=False)
    cp, y0 = navier_stokes_cavity(16, re=100.0)
    y0 = y0 + 0.0
    y0[1:-1, 1:-1, 0] = np.random.RandomState(steps).uniform(-1, 1, (15, 15))
    ivp = pml.InitialValueProblem(cp, (0.0, steps * 1e-4),
                                  pml.DiscreteInitialCondition(cp, y0, True))

    def solve(limit):
        diff = ThreePointCentralDifferenceMethod(tol=1e-4, max_sweeps=limit)
        op = FDMOperator(RK4(), diff, 1e-4, precision=precision, snapshot_every=every)
        return op.solve(ivp).discrete_y()

    want = solve(16383)  # a limit of the caller's own: stepped from the host
    lib = _Library(nat.device_lib(), fails_at)
    monkeypatch.setattr(nat, "device_lib", lambda: lib)
    assert np.array_equal(solve(10_000_000), want)
    assert lib.single == single
