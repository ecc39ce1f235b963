"""x ** 1.5 at the ends of the number line as pow gives it, in both ways a
program runs: per vertex (``pml_expr_eval``) and as an ODE system in the lanes
of a wavefront and on one thread (``pml_ode_solve``)."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VALUES = [np.inf, -np.inf, 0.0, -0.0, -1.0, np.nan, 4.0]


@pytest.mark.parametrize("precision", ["float64", "float32"])
def test_limits_of_the_three_halves_power(precision):
    import sympy as sp
    import torch

    from pararealml_amd import _native as nat
    from pararealml_amd.operators.device_program import compile_expressions

    print(f"case: three-halves limits {precision}", flush=True)
    prec = nat.PML_F64 if precision == "float64" else nat.PML_F32
    big = 1e200 if precision == "float64" else 1e30  # its power overflows
    x = np.array(VALUES + [big, np.finfo(precision).max, np.finfo(precision).tiny], precision)
    with np.errstate(all="ignore"):
        want = np.power(x, x.dtype.type(1.5))
    s = sp.Symbol("x")
    program = compile_expressions([s**sp.Rational(3, 2)], lambda _: 0, [s])
    lib, st = nat.device_lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    y = torch.from_numpy(x).cuda()
    out = torch.empty_like(y)
    nat.check(lib.pml_expr_eval(
        prec, program.handle(), (ctypes.c_void_p * 1)(y.data_ptr()), (ctypes.c_int64 * 1)(1),
        (ctypes.c_void_p * 1)(out.data_ptr()), (ctypes.c_int64 * 1)(1), 0.0, len(x), st))
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    # one Euler step y + y ** 1.5, far below and above the batch of one thread a system
    with np.errstate(all="ignore"):
        want = x + want
    for repeats in (1, 1000):
        z = y.repeat(repeats)
        batch = len(z)
        zeros = torch.zeros(batch, dtype=torch.float64, device="cuda")
        nat.check(lib.pml_ode_solve(prec, program.handle(), nat.PML_INT_FE, batch,
                                    zeros.data_ptr(), zeros.data_ptr(), 1.0, 1, z.data_ptr(),
                                    None, 0, st))
        np.testing.assert_array_equal(z[:len(x)].cpu().numpy(), want)
