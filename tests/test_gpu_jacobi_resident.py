"""The Jacobi loop that runs in one workgroup against the loop of one launch
per sweep (``pml_jacobi_sweep``): the same iterates and sweep counts, at the
edges of its sizes (vertices a thread, the largest grid) and one vertex beside
them, on lines, plates and boxes, for several fields, with and without
constraints (plates between fixed edges up to their largest); its exits (a sweep limit, values that are not numbers); and the
Navier-Stokes time loop around it against stepping from the host."""

import ctypes

import numpy as np
import pytest

from tests.helpers import navier_stokes_cavity

pytestmark = pytest.mark.gpu

# (shape, fields): up to 2 and 5 values a thread of 1024, one beside them, and
# grids that two launches a sweep take
SIZES = [((3,), 1), ((3, 3), 2), ((1025,), 1), ((32, 64), 1), ((17, 11, 11), 1),
         ((64, 80), 1), ((64, 81), 1), ((29, 23, 13), 2), ((138, 133), 1), ((135, 137), 1)]


def _setup(shape, fields, dtype, constrained):
    import torch

    rng = np.random.RandomState(sum(shape))
    full = tuple(shape) + (1,) * (3 - len(shape))
    dx = [0.1, 0.125, 0.2][:len(shape)] + [1.0] * (3 - len(shape))
    y = torch.from_numpy(rng.uniform(-1, 1, full + (fields,))).to("cuda", dtype)
    lap = torch.from_numpy(rng.uniform(-1, 1, full + (fields,))).to("cuda", dtype)
    fixed = ghosts = None
    lo, hi = [None] * 3, [None] * 3
    if constrained:
        fixed = torch.full(full + (fields,), float("nan"), dtype=torch.float64, device="cuda")
        fixed[0] = 0.25
        y[0] = 0.25
        slab = int(np.prod(full)) // shape[-1] * fields
        axis = len(shape) - 1
        hi[axis] = torch.from_numpy(rng.uniform(-1, 1, slab)).cuda()
        lo[axis] = torch.full((slab,), float("nan"), dtype=torch.float64, device="cuda")
    ptr = lambda a: None if a is None else a.data_ptr()  # noqa: E731
    c = dict(shape=(ctypes.c_int64 * 3)(*full), dx=(ctypes.c_double * 3)(*dx),
             lo=(ctypes.c_void_p * 3)(*[ptr(a) for a in lo]),
             hi=(ctypes.c_void_p * 3)(*[ptr(a) for a in hi]), fixed=ptr(fixed),
             keep=(lo, hi, fixed))
    return y, lap, c


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("constrained", [False, True])
@pytest.mark.parametrize("shape,fields", SIZES)
def test_resident_loop_equals_the_sweeps(shape, fields, constrained, precision):
    import torch

    from pararealml_amd import _native as nat

    print(f"case: resident jacobi {shape} x {fields} {constrained} {precision}", flush=True)
    prec = nat.PML_F64 if precision == "float64" else nat.PML_F32
    dtype = torch.float64 if precision == "float64" else torch.float32
    lib = nat.device_lib()
    y, lap, c = _setup(shape, fields, dtype, constrained)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    work = torch.zeros(nat.PML_REDUCE_SLOTS, dtype=torch.float64, device="cuda")
    norm = torch.zeros(1, dtype=torch.float64, device="cuda")
    want, norms = y.clone(), []
    for _ in range(12):
        new = torch.empty_like(want)
        nat.check(lib.pml_jacobi_sweep(prec, want.data_ptr(), new.data_ptr(), lap.data_ptr(),
                                       c["shape"], fields, c["dx"], c["lo"], c["hi"], c["fixed"],
                                       norm.data_ptr(), work.data_ptr(), st))
        want = new
        norms.append(float(norm) ** 0.5)
    tol = 1.0000001 * min(norms)  # reached by sweep k, and by none before it
    k = 1 + next(i for i, v in enumerate(norms) if v <= tol)
    state = torch.zeros(nat.PML_JACOBI_STATE_BYTES // 8, dtype=torch.float64, device="cuda")
    sweeps, diff = ctypes.c_int64(0), ctypes.c_double(0.0)

    def solve(start, tol, limit):
        cur, spare = start.clone(), torch.empty_like(start)
        nat.check(lib.pml_jacobi_solve(
            prec, cur.data_ptr(), spare.data_ptr(), lap.data_ptr(), c["shape"], fields, c["dx"],
            c["lo"], c["hi"], c["fixed"], tol, limit, 64, state.data_ptr(),
            ctypes.byref(sweeps), ctypes.byref(diff), st))
        return cur

    got = solve(y, tol, 1000)
    assert sweeps.value == k
    assert diff.value == pytest.approx(norms[k - 1], rel=1e-12)
    if k == 12:
        assert torch.equal(got, want)
    got = solve(y, 0.0, 12)  # the sweep limit: the last iterate, reported as unfinished
    assert sweeps.value == -12 and torch.equal(got, want)
    bad = y.clone().view(-1)
    bad[-1] = float("nan")
    solve(bad.view_as(y), 1e-3, 40)
    assert sweeps.value == -40 and np.isnan(diff.value)


# between fixed edges: 5 and up to 18 vertices a thread, the largest plates of
# each precision and those beside them; in one workgroup in FP64, in FP32
PLATES = [((64, 80), True, True), ((65, 79), True, True), ((100, 103), True, True),
          ((124, 128), True, True), ((125, 129), False, True), ((128, 144), False, True),
          ((129, 144), False, False)]


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("shape,f64,f32", PLATES)
def test_resident_plates_between_fixed_edges(shape, f64, f32, precision):
    import torch

    from pararealml_amd import _native as nat

    print(f"case: resident plate {shape} {precision}", flush=True)
    prec = nat.PML_F64 if precision == "float64" else nat.PML_F32
    dtype = torch.float64 if precision == "float64" else torch.float32
    lib = nat.device_lib()
    y, lap, c = _setup(shape, 1, dtype, False)
    fixed = torch.full(shape, float("nan"), dtype=torch.float64, device="cuda")
    fixed[0], fixed[-1], fixed[:, 0], fixed[:, -1] = 0.25, -0.5, 0.125, 1.0
    y = torch.where(fixed.isnan(), y.view(shape), fixed.to(dtype))
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    work = torch.zeros(nat.PML_REDUCE_SLOTS, dtype=torch.float64, device="cuda")
    norm = torch.zeros(1, dtype=torch.float64, device="cuda")
    want = y.clone()
    for _ in range(9):
        new = torch.empty_like(want)
        nat.check(lib.pml_jacobi_sweep(prec, want.data_ptr(), new.data_ptr(), lap.data_ptr(),
                                       c["shape"], 1, c["dx"], c["lo"], c["hi"],
                                       fixed.data_ptr(), norm.data_ptr(), work.data_ptr(), st))
        want = new
    # the loop of two launches leaves its partial sums here
    state = torch.full((nat.PML_JACOBI_STATE_BYTES // 8,), -1.0, dtype=torch.float64,
                       device="cuda")
    sweeps, diff = ctypes.c_int64(0), ctypes.c_double(0.0)
    spare = torch.empty_like(y)
    nat.check(lib.pml_jacobi_solve(
        prec, y.data_ptr(), spare.data_ptr(), lap.data_ptr(), c["shape"], 1, c["dx"], c["lo"],
        c["hi"], fixed.data_ptr(), 0.0, 9, 64, state.data_ptr(), ctypes.byref(sweeps),
        ctypes.byref(diff), st))
    assert sweeps.value == -9 and torch.equal(y, want)
    assert bool((state[4:] == -1.0).all()) == (f64 if precision == "float64" else f32)


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("n,tol", [(8, 1e-3), (33, 1e-4), (64, 1e-6), (160, 1e-3)])
def test_poisson_time_loop_equals_stepping_from_the_host(n, tol, precision, monkeypatch):
    import pararealml_amd as pml
    from pararealml_amd.operators.fdm import (
        RK4, FDMOperator, ForwardEulerMethod, ThreePointCentralDifferenceMethod)

    loop, taken = FDMOperator._poisson_loop, []  # the steps that the device loop took

    def recorded(self, *args):
        taken.append(loop(self, *args))
        return taken[-1]

    monkeypatch.setattr(FDMOperator, "_poisson_loop", recorded)

    print(f"case: poisson loop {n} {tol} {precision}", flush=True)
    cp, y0 = navier_stokes_cavity(n, re=100.0)
    y0 = y0 + 0.0
    y0[1:-1, 1:-1, 0] = np.random.RandomState(n).uniform(-1, 1, (n - 1, n - 1))
    ivp = pml.InitialValueProblem(cp, (0.0, 5e-4), pml.DiscreteInitialCondition(cp, y0, True))
    for integrator in (ForwardEulerMethod(), RK4()):
        outs = []
        taken.clear()
        # a sweep limit of the caller's own takes the host's loop
        for limit in (10_000_000, 16383):
            diff = ThreePointCentralDifferenceMethod(tol=tol, max_sweeps=limit)
            op = FDMOperator(integrator, diff, 1e-4, precision=precision)
            outs.append((op.solve(ivp).discrete_y(), diff.last_jacobi_sweeps))
        assert outs[0][1] == outs[1][1] > 0
        assert np.array_equal(outs[0][0], outs[1][0])
        # a grid of 161 x 161 is beyond one workgroup
        assert taken == [5 if n < 160 else 0, 0]
