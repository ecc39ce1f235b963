"""The ODE kernel that runs a program's independent instructions in the lanes
of one wavefront per system, against the kernel of one thread per system
(which a batch above the wavefront kernel's limit takes): the same operations,
so the same bits, for systems with more than 64 independent instructions, with
every kind of instruction, and with one variable.  The limit is 256 systems per
instruction of the program, 64 with elementary functions, and lower where the
instructions wait for one another."""

import ctypes

import numpy as np
import pytest

import pararealml_amd as pml
from pararealml_amd.differential_equation import DifferentialEquation, SymbolicEquationSystem

pytestmark = pytest.mark.gpu


class _Decay(DifferentialEquation):
    def __init__(self):
        super().__init__(0, 1)

    @property
    def symbolic_equation_system(self):
        return SymbolicEquationSystem([-self.symbols.y[0] * (1.0 + self.symbols.t) ** 3])


class _EveryKind(DifferentialEquation):
    def __init__(self):
        super().__init__(0, 4)

    @property
    def symbolic_equation_system(self):
        import sympy as sp

        a, b, c, d = self.symbols.y
        t = self.symbols.t
        return SymbolicEquationSystem([
            sp.sin(a) * sp.cos(t) - sp.Abs(b) ** sp.Rational(3, 2) + sp.exp(-c**2) + a**-2,
            sp.sqrt(1 + a**2) * sp.tanh(b) - sp.Max(c, d) + sp.Min(a, b, 0.3),
            sp.atan2(a, 1 + b**2) + sp.log(2 + c**2) - (1 + d**2) ** 0.3 + sp.sign(a) * 0.1,
            (a * b - c / (1 + d**2)) / 3 + sp.atan(a) - sp.sinh(b) * sp.cosh(c) * 0.01,
        ])


def _system(name):
    if name == "one":
        return _Decay(), np.array([1.25])
    if name == "kinds":
        return _EveryKind(), np.array([0.7, -0.4, 0.9, 0.2])
    if name == "lorenz":
        return pml.LorenzEquation(), np.array([1.0, 1.1, 0.9])
    k = int(name[-1])
    rng = np.random.RandomState(k)
    pos = rng.uniform(-0.2, 0.2, (k, 3)) + 2.0 * np.arange(k)[:, None]
    return (pml.NBodyGravitationalEquation(3, list(rng.uniform(0.5, 2.0, k)), g=1.0),
            np.concatenate([pos.ravel(), rng.uniform(-0.3, 0.3, 3 * k)]))


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("name", ["one", "kinds", "lorenz", "bodies-2", "bodies-5"])
def test_wave_schedule_equals_the_serial_program(name, precision):
    import torch

    from pararealml_amd import _native as nat
    from pararealml_amd.operators.device_program import ode_program

    eq, y0 = _system(name)
    program, n = ode_program(eq), len(y0)
    prec = nat.PML_F64 if precision == "float64" else nat.PML_F32
    dtype = torch.float64 if precision == "float64" else torch.float32
    lib = nat.device_lib()
    for integ in (nat.PML_INT_FE, nat.PML_INT_MIDPOINT, nat.PML_INT_RK4):
        outs = []
        # (the limit is at most 256 systems per instruction)
        for batch in (3, 256 * len(program.code) + 1):
            print(f"case: ode wave {name} {precision} {integ} batch {batch}", flush=True)
            assert (lib.pml_ode_wave_rounds(program.handle(), batch) > 0) == (batch == 3)
            scale = 1.0 + 0.01 * torch.arange(batch, dtype=torch.float64).remainder(3)
            y = (torch.from_numpy(y0)[None] * scale[:, None]).to("cuda", dtype).contiguous()
            t0 = (0.25 * torch.arange(batch, dtype=torch.float64).remainder(3)).cuda()
            step = torch.full((batch,), 1e-2, dtype=torch.float64, device="cuda")
            snaps = torch.empty((3, batch, n), dtype=dtype, device="cuda")
            nat.check(lib.pml_ode_solve(
                prec, program.handle(), integ, batch, t0.data_ptr(), step.data_ptr(), 1e-2, 7,
                y.data_ptr(), snaps.data_ptr(), 2,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
            outs.append((y[:3].cpu().numpy(), snaps[:, :3].cpu().numpy()))
        assert np.all(np.isfinite(outs[0][0]))
        assert np.array_equal(outs[0][0], outs[1][0])
        assert np.array_equal(outs[0][1], outs[1][1])


def test_three_halves_power():
    """x ** 1.5 within one rounding of the exact value in FP64 (80-bit
    reference), and the limits of pow."""
    import sympy as sp
    import torch

    from pararealml_amd import _native as nat
    from pararealml_amd.operators.device_program import compile_expressions

    print("case: three-halves power", flush=True)
    x = np.concatenate([np.random.RandomState(0).uniform(0.0, 8.0, 4000),
                        10.0 ** np.random.RandomState(1).uniform(-180, 180, 4000),
                        [0.0, np.inf, -1.0, np.nan]])
    s = sp.Symbol("x")
    program = compile_expressions([s**sp.Rational(3, 2)], lambda _: 0, [s])
    y, out = torch.from_numpy(x).cuda(), torch.empty(len(x), dtype=torch.float64, device="cuda")
    nat.check(nat.device_lib().pml_expr_eval(
        nat.PML_F64, program.handle(), (ctypes.c_void_p * 1)(y.data_ptr()),
        (ctypes.c_int64 * 1)(1), (ctypes.c_void_p * 1)(out.data_ptr()), (ctypes.c_int64 * 1)(1),
        0.0, len(x), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = out.cpu().numpy()
    ref = x[:-4].astype(np.longdouble)
    ref = ref * np.sqrt(ref)
    # one FP64 rounding plus the compensated tail's second-order error
    assert np.max(np.abs(got[:-4] - ref) / ref) <= 0.52 * 2.0**-52
    assert got[-4] == 0.0 and np.isposinf(got[-3]) and np.isnan(got[-2]) and np.isnan(got[-1])


def _nested(depth, width, f):
    class Nested(DifferentialEquation):
        def __init__(self):
            super().__init__(0, width)

        @property
        def symbolic_equation_system(self):
            out = []
            for v in self.symbols.y:
                for _ in range(depth):
                    v = f(v)
                out.append(v)
            return SymbolicEquationSystem(out)

    return Nested()


@pytest.mark.parametrize("name,lanes,serial", [
    # systems at once that run in lanes, and that run one a thread
    ("roots-40", (1, 256), (1024, 5312, 21248)),
    ("roots-10", (1, 256, 1024), (5888,)),
    ("squares-40", (1, 1024), (5312, 21248)),
    ("sines-40", (1, 256, 1024), (2688,)),
    ("horner", (1, 1024, 2048), (4096,)),
    ("lorenz", (1, 1024, 4608), (4609,)),
    ("bodies-2", (1, 4096), (16384,)),
])
def test_deep_programs_share_out_less(name, lanes, serial):
    import sympy as sp

    from pararealml_amd import _native as nat
    from pararealml_amd.operators.device_program import ode_program

    print(f"case: ode route {name}", flush=True)
    kind, _, depth = name.partition("-")
    f = {"roots": lambda v: sp.sqrt(v + 2), "squares": lambda v: v**2 - sp.Rational(1, 3),
         "sines": sp.sin}.get(kind)
    if f is not None:
        eq = _nested(int(depth), 1, f)
    elif kind == "horner":
        eq = _nested(1, 1, lambda y: ((((y / 2 + 1) * y - 2) * y + sp.Rational(3, 10)) * y
                                      - sp.Rational(1, 10)) * y)
    else:
        eq = _system(name)[0]
    program, lib = ode_program(eq), nat.device_lib()
    for batch in lanes:
        assert lib.pml_ode_wave_rounds(program.handle(), batch) > 0, batch
    for batch in serial:
        assert lib.pml_ode_wave_rounds(program.handle(), batch) == 0, batch
