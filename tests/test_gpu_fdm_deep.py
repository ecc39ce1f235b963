"""The many-step kernel (PML_FLAG_AUTO) against the default streaming variant:
equal to the bit for every equation, integrator and precision, on grids that
fit one region, that need tiles with halos and that lie beside multiples of
both (down to 3 vertices an axis), on lines, on ragged batches, with snapshots
every step, at intervals that do not divide a launch's steps and without,
Dirichlet and Neumann edges mixed per side, the input constrained in the call."""

import ctypes

import numpy as np
import pytest

import pararealml_amd as pml
from pararealml_amd import _native as nat

pytestmark = pytest.mark.gpu

EQUATIONS = {
    "diffusion": lambda nd: pml.DiffusionEquation(nd, 0.4),
    "convection_diffusion": lambda nd: pml.ConvectionDiffusionEquation(
        nd, [0.3, -0.2][:nd], 0.05),
    "wave": lambda nd: pml.WaveEquation(nd, 1.1),
    "burgers": lambda nd: pml.BurgersEquation(nd, 50.0),
    "shallow_water": lambda nd: pml.ShallowWaterEquation(h=1.0, b=0.02, v=0.03, f=0.1, g=9.81),
    "cahn_hilliard": lambda nd: pml.CahnHilliardEquation(nd, 0.1, 0.01),
}
D_X, D_T = 0.1, 1e-4


def _problem(name, shape):
    from pararealml_amd import _device as dev

    eq = EQUATIONS[name](len(shape))
    f = eq.y_dimension
    mesh = pml.Mesh([(0.0, D_X * (n - 1)) for n in shape], [D_X] * len(shape))
    dirichlet = pml.DirichletBoundaryCondition(
        lambda x, t: np.stack([0.1 * (k + 1) + 0.2 * x[:, 0] for k in range(f)], axis=-1),
        is_static=True)
    neumann = pml.NeumannBoundaryCondition(
        lambda x, t: np.stack([0.3 * (k - 1) + 0.1 * x[:, -1] for k in range(f)], axis=-1),
        is_static=True)
    pairs = [(dirichlet, neumann), (neumann, dirichlet)]
    return dev.device_problem(pml.ConstrainedProblem(eq, mesh, pairs[:len(shape)]))


def _steps_a_launch(batch, steps):
    """0: the streaming kernels run the batch."""
    plan = (ctypes.c_int * 4)()
    nat.check(batch.lib.pml_fdm_auto_plan(batch.eq_id, batch.integrator, batch.prec, batch.ndim,
                                          batch.grids, len(batch.grid_problem), steps, plan))
    return plan[3]


def _compare(name, shapes, integ, precision, steps, every, taken=True):
    import torch

    from pararealml_amd import _device as dev

    print(f"case: deep {name} {shapes} {integ} {precision} {steps}/{every}", flush=True)
    problems = [_problem(name, s) for s in shapes]
    rng = np.random.RandomState(len(shapes) + steps)
    ys = [rng.uniform(-0.5, 0.5, tuple(s) + (p.n_fields,)) for s, p in zip(shapes, problems)]
    stream = dev.solver_stream()
    outs = []
    with torch.cuda.stream(stream):
        for auto in (False, True):
            b = dev.FDMBatch(problems, list(range(len(shapes))), precision, integ, stream)
            assert (_steps_a_launch(b, steps) > 0) == taken
            b.load_host(ys)
            snaps = b.new_snapshots(steps // every) if every else None
            b.advance(D_T, steps, snaps, every, constrain_input=True, auto=auto)
            outs.append([b.state_f64().cpu().numpy()]
                        + ([b.snapshots_f64(snaps, steps // every).cpu().numpy()]
                           if every else []))
    assert np.all(np.isfinite(outs[0][0]))
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["float64", "float32", "float32c"])
@pytest.mark.parametrize("integ", [0, 1, 2])
@pytest.mark.parametrize("name", list(EQUATIONS))
def test_many_step_kernel_equals_the_streaming_one(name, integ, precision):
    _compare(name, [(3, 3)], integ, precision, 5, 1)  # one region
    _compare(name, [(31, 33)], integ, precision, 10, 0)  # 1023 vertices
    _compare(name, [(33, 33)], integ, precision, 9, 3)
    _compare(name, [(48, 65)], integ, precision, 22, 11)  # tiles, rows and columns of one vertex
    _compare(name, [(200, 131)], integ, precision, 19, 1)
    _compare(name, [(3, 700)], integ, precision, 7, 7)


@pytest.mark.parametrize("precision", ["float64", "float32c"])
@pytest.mark.parametrize("name", ["diffusion", "convection_diffusion", "wave", "burgers"])
@pytest.mark.parametrize("n", [3, 64, 255, 449, 1025, 2049, 5000])
def test_many_step_kernel_on_lines(name, n, precision):
    for integ in (0, 2):
        _compare(name, [(n,)], integ, precision, 100, 50 if n % 2 else 0)


def test_many_step_kernel_on_ragged_batches():
    for precision in ("float64", "float32"):
        _compare("cahn_hilliard", [(20, 33), (64, 40), (3, 5), (97, 24)], 2, precision, 12, 4)
        _compare("shallow_water", [(33, 20), (64, 64), (41, 97)], 2, precision, 6, 1)
    _compare("burgers", [(90,), (300,), (7,)], 1, "float64", 12, 6)


def test_large_batches_keep_their_variant():
    _compare("diffusion", [(700, 700)], 2, "float32", 3, 0, taken=False)  # above 640 tiles


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("integ", [0, 1, 2])
@pytest.mark.parametrize("n", [4, 31, 65, 129])
def test_navier_stokes_single_steps(n, integ, precision):
    """The step inside a Poisson time loop: algebraic fields, one step a
    launch; and several, which no rule on short runs keeps from the kernel."""
    import torch

    from pararealml_amd import _device as dev
    from tests.helpers import navier_stokes_cavity

    print(f"case: deep navier-stokes {n} {integ} {precision}", flush=True)
    cp, y0 = navier_stokes_cavity(n, re=100.0)
    y0 = y0 + np.random.RandomState(n).uniform(-0.5, 0.5, y0.shape)
    problem = dev.device_problem(cp)
    stream = dev.solver_stream()
    outs = []
    with torch.cuda.stream(stream):
        for auto in (False, True):
            b = dev.FDMBatch([problem], [0], precision, integ, stream, poisson_phase=True)
            b.load_host([y0])
            assert _steps_a_launch(b, 3) > 0
            for steps in (1, 1, 1, 3):
                b.advance(D_T, steps, auto=auto)
            outs.append(b.state_f64().cpu().numpy())
    assert np.all(np.isfinite(outs[0])) and np.array_equal(*outs)
