"""Tuning and the many-step kernel: the tuner times it as one more candidate
where it has a plan for the batch, and a recorded variant turns it off only
where it was timed and slower."""

import ctypes
import json

import numpy as np
import pytest

import pararealml_amd as pml
from pararealml_amd import _native as nat
from pararealml_amd import autotune


@pytest.fixture
def fresh_cache(tmp_path, monkeypatch):
    path = tmp_path / "tune.json"
    monkeypatch.setenv("PML_AUTOTUNE_CACHE", str(path))
    monkeypatch.setattr(autotune, "_cache", None)
    yield path
    autotune._cache = None


def _operator(n=33, **kw):
    from pararealml_amd.operators.fdm import RK4, FDMOperator, ThreePointCentralDifferenceMethod

    mesh = pml.Mesh([(0.0, 1.0)] * 2, [1.0 / (n - 1)] * 2)
    bc = pml.DirichletBoundaryCondition(lambda x, t: np.zeros((len(x), 1)), is_static=True)
    cp = pml.ConstrainedProblem(pml.DiffusionEquation(2, 0.5), mesh, [(bc, bc), (bc, bc)])
    return FDMOperator(RK4(), ThreePointCentralDifferenceMethod(), 1e-5, **kw), cp


def _plan(eq, integ, prec, shapes, n_steps):
    grids = (nat.PmlGrid * len(shapes))()
    for g, s in zip(grids, shapes):
        g.n0, g.n1 = (1,) * (2 - len(s)) + tuple(s)
        g.dx0 = g.dx1 = 0.1
    out = (ctypes.c_int * 4)()
    nat.check(nat.load_library().pml_fdm_auto_plan(
        nat.PML_EQ[eq], integ, prec, len(shapes[0]), grids, len(shapes), n_steps, out))
    return tuple(out)


def test_plans_of_the_many_step_kernel():
    """(output rows, columns, halo, steps a launch), 0 where the streaming
    kernels run the batch; no GPU needed."""
    rk4, f64, f32 = nat.PML_INT_RK4, nat.PML_F64, nat.PML_F32
    assert _plan("diffusion", rk4, f64, [(33, 33)], 100) == (33, 33, 0, 100)
    assert _plan("diffusion", rk4, f64, [(33, 33)], 5000)[3] == 2048
    rows, columns, halo, steps = _plan("diffusion", rk4, f32, [(300, 300)], 64)
    assert halo == 4 * steps > 0 and 300 > rows == columns
    assert _plan("burgers", rk4, f64, [(5000,)], 48)[0] == 1
    assert _plan("diffusion", rk4, f32, [(700, 700)], 64) == (0, 0, 0, 0)
    assert _plan("diffusion", rk4, f32, [(33, 33)] * 641, 64) == (0, 0, 0, 0)
    assert _plan("diffusion", rk4, f64, [(33, 33)], 0) == (0, 0, 0, 0)
    assert nat.load_library().pml_fdm_auto_plan(0, 0, 0, 3, None, 0, 1, None) == nat.PML_E_INVALID


@pytest.mark.parametrize("entry,config,auto", [
    (None, 0, True),
    ("{last}", -1, True),  # recorded without a timing of the many-step kernel
    ("{last} < many-step", -1, False),
    ("{last} > many-step", -1, True),
    ("pruned-variant", 0, True),
    ("pruned-variant < many-step", 0, True),
])
def test_recorded_variants_and_the_many_step_kernel(fresh_cache, monkeypatch, entry, config, auto):
    from pararealml_amd import _device as dev

    op, cp = _operator()
    problem = dev.device_problem(cp)
    names = autotune.variant_names(nat.PML_EQ["diffusion"], nat.PML_INT_RK4, nat.PML_F64)
    if entry is not None:
        key = autotune.key_for(problem, nat.PML_INT_RK4, "float64")
        fresh_cache.write_text(json.dumps({key: entry.format(last=names[-1])}))
    assert op.kernel_choice(problem) == dict(tile_config=config % len(names), auto=auto)
    given, _ = _operator(tile_config=1)
    assert given.kernel_choice(problem) == dict(tile_config=1, auto=False)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["float64", "float32", "float32c"])
def test_tuning_times_the_many_step_kernel(fresh_cache, monkeypatch, precision):
    print(f"case: tune many-step {precision}", flush=True)
    seen = []
    tune = autotune.tune
    monkeypatch.setattr(autotune, "tune", lambda *a, **k: seen.append(tune(*a, **k)) or seen[-1])
    op, cp = _operator(precision=precision)
    problem = op.device_problem(cp)
    best = op.tune(cp, n_steps=64)
    timings = seen[0][1]
    streaming = [v for k, v in timings.items() if k != "many-step"]
    names = [k for k in timings if k != "many-step"]
    assert names[best] == min(names, key=timings.get)
    assert op.kernel_choice(problem) == dict(
        tile_config=best, auto=timings["many-step"] < min(streaming))
    # 33 x 33 vertices are a few microseconds a step for a launch, and one to
    # two for the steps of a launch
    assert op.kernel_choice(problem)["auto"]
    op.tune(cp, n_grids=700, n_steps=2)  # no plan: nothing to time
    assert "many-step" not in seen[1][1]
