"""Which runs the fused time loop of the diffusion equation takes: those
``pml_laplacian_solve`` accepts; larger grids stay on the composed loop, whose
kernels index in 64 bits."""

import ctypes

import numpy as np
import pytest

import pararealml_amd as pml
from pararealml_amd import _native as nat
from pararealml_amd.operators.fdm import FDMOperator, ForwardEulerMethod
from pararealml_amd.operators.fdm import ThreePointCentralDifferenceMethod as Central


def _accepted(shape):
    """What the library says of a run of no steps (nothing is launched)."""
    full = tuple(shape) + (1,) * (3 - len(shape))
    some = ctypes.create_string_buffer(8)
    rc = nat.load_library().pml_laplacian_solve(
        nat.PML_F64, nat.PML_INT_FE, (ctypes.c_int64 * 3)(*full), (ctypes.c_double * 3)(1, 1, 1),
        None, None, 1, (ctypes.c_int * 1)(0), (ctypes.c_int * 1)(2), None, None, 1.0, 1.0, 0,
        some, some, ctypes.cast(some, ctypes.c_void_p), 1, None)
    assert rc in (nat.PML_OK, nat.PML_E_INVALID)
    return rc == nat.PML_OK


@pytest.mark.parametrize("shape", [
    (33, 29, 31), (2**31 - 256,), (2**31 - 255,), (1290, 1290, 1290), (1291, 1291, 1291),
    (1300, 1300, 1300), (46340, 46340), (46341, 46341), (3, 2**31 // 3), (65536, 65536, 4),
])
def test_grids_of_the_fused_loop(shape):
    assert Central.takes_laplacian_solve(shape) == _accepted(shape)


def test_boxes_of_more_axes_stay_on_the_composed_loop():
    assert not Central.takes_laplacian_solve((4, 4, 4, 4))


@pytest.mark.gpu
def test_composed_loop_equals_the_fused_one(monkeypatch):
    print("case: laplacian route", flush=True)
    mesh = pml.Mesh([(0.0, 1.0)] * 3, [0.125, 0.25, 0.2])
    bc = pml.DirichletBoundaryCondition(lambda x, t: 0.1 + x[:, :1], is_static=True)
    free = pml.NeumannBoundaryCondition(lambda x, t: x[:, 1:2], is_static=True)
    cp = pml.ConstrainedProblem(pml.DiffusionEquation(3, 0.3), mesh, [(bc, free)] * 3)
    y0 = np.random.RandomState(3).uniform(-1.0, 1.0, cp.y_vertices_shape)
    ivp = pml.InitialValueProblem(cp, (0.0, 6e-3), pml.DiscreteInitialCondition(cp, y0, True))
    calls = []
    fused = Central.solve_laplacian
    monkeypatch.setattr(Central, "solve_laplacian",
                        lambda *a, **k: calls.append(1) or fused(*a, **k))
    op = FDMOperator(ForwardEulerMethod(), Central(), 1e-3)
    want = op.solve(ivp).discrete_y()
    assert calls == [1]
    monkeypatch.setattr(Central, "LAPLACIAN_SOLVE_VERTICES", int(np.prod(mesh.vertices_shape)) - 1)
    got = op.solve(ivp).discrete_y()
    assert calls == [1] and np.array_equal(got, want)
