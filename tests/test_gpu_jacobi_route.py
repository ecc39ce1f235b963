"""Which plates the Jacobi iteration keeps in one workgroup: by the measured
cost of a sweep there, which grows with the free vertices on the edges,
against that of two launches.  The loop of two launches leaves its partial
sums in the state buffer, the loop in one workgroup does not touch them."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (rows, columns, fixed edges, in one workgroup in FP64, in FP32)
PLATES = [
    (17, 17, "none", True, True), (65, 65, "none", True, True), (65, 65, "null", True, True),
    (90, 90, "null", False, False), (90, 90, "all", True, True),
    (100, 100, "none", False, False), (100, 100, "null", False, False),
    (100, 100, "rows", False, False), (100, 100, "one column", False, False),
    (100, 100, "columns", True, True), (100, 100, "all", True, True),
    (129, 129, "none", False, False), (129, 129, "all", False, True),
    (400, 20, "none", False, False), (400, 20, "columns", True, True),
    (32, 256, "rows", False, False), (32, 256, "all", True, True),
    (135, 137, "all", False, False),
]


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("n0,n1,edges,f64,f32", PLATES)
def test_plates_in_one_workgroup(n0, n1, edges, f64, f32, precision):
    import torch

    from pararealml_amd import _native as nat

    print(f"case: jacobi route {n0} x {n1} {edges} {precision}", flush=True)
    prec = nat.PML_F64 if precision == "float64" else nat.PML_F32
    dtype = torch.float64 if precision == "float64" else torch.float32
    rng = np.random.RandomState(n0)
    y = torch.from_numpy(rng.uniform(-1.0, 1.0, (n0, n1))).to("cuda", dtype)
    lap, spare = torch.zeros_like(y), torch.empty_like(y)
    fixed = torch.full((n0, n1), float("nan"), dtype=torch.float64, device="cuda")
    if edges in ("rows", "all"):
        fixed[0] = fixed[-1] = 0.5
    if edges in ("columns", "all"):
        fixed[:, 0] = fixed[:, -1] = 0.5
    if edges == "one column":
        fixed[:, 0] = 0.5
    state = torch.full((nat.PML_JACOBI_STATE_BYTES // 8,), -1.0, dtype=torch.float64,
                       device="cuda")
    sweeps, diff = ctypes.c_int64(0), ctypes.c_double(0.0)
    none = (ctypes.c_void_p * 3)()
    nat.check(nat.device_lib().pml_jacobi_solve(
        prec, y.data_ptr(), spare.data_ptr(), lap.data_ptr(), (ctypes.c_int64 * 3)(n0, n1, 1), 1,
        (ctypes.c_double * 3)(0.1, 0.1, 1.0), none, none,
        None if edges == "null" else fixed.data_ptr(), 0.0, 3, 64, state.data_ptr(),
        ctypes.byref(sweeps), ctypes.byref(diff),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert sweeps.value == -3
    assert bool((state[4:] == -1.0).all()) == (f64 if precision == "float64" else f32)
