"""Parareal on one GPU.

``PararealOperator(f, g, termination_condition, max_iterations)`` keeps the
reference's interface and algorithm (pararealml/operators/parareal/
parareal_operator.py:13-197) with the time slices as the batch axis of one
device tensor instead of MPI ranks:

1. the slice length is ``(t1 - t0) / n_slices`` and must be a multiple of
   both operators' time steps (the reference's ``ValueError`` checks);
2. the coarse operator sweeps the slices once from the initial value;
3. each iteration i runs the fine solves of slices i..N-1 together (slices
   before i have unchanged initial values, so their fine results would be
   identical), forms the FP64 corrections ``F_end - G_end``, then sweeps
   slices i..N-1 serially: ``G_end[j] = g(U[j])`` for j > i and
   ``U[j+1] = G_end[j] + corr[j]``, accumulating the per-field squared
   updates;
4. it stops when, for every field, the maximum over slices of the RMS
   update is below the tolerance (or a callable ``termination_condition``
   says so), or after ``min(n_slices, max_iterations)`` iterations;
5. the output is each slice's last fine trajectory shifted by
   ``U[r+1] - F_r[-1]``.

The border points U, the coarse end points, the corrections and the update
norms are FP64 in HBM; the fine and coarse states use their operators'
precisions.  ``n_slices`` replaces the MPI communicator size;
``output="endpoints"`` returns only the slice end points (the full fine
trajectory is infeasible for long runs).  The iteration count and timings
of the last solve are in ``last_iterations`` and ``last_stats``; an optional
``monitor(iteration, u)`` is called after every iteration with the FP64
border points ``u`` (device tensor, (N + 1, elems), field-major), its time is
excluded from the timings, and a True return ends the iterations.

``coarse_increments=True`` evaluates the coarse propagator on the change of
each slice's initial value instead of on the new and the old value:
``U_new[j+1] = F(U_old[j]) + G(U_new[j] - U_old[j])``, which equals the
reference's ``G(U_new[j]) + F(U_old[j]) - G(U_old[j])`` for a linear coarse
propagator (the equation linear, the boundary values homogeneous; both are
checked).  For a learned coarse propagator whose network normalises its
input by the input's own magnitude, it is the form in which the network
resolves the iterates' small changes at all: evaluated on the states, a
change of 1e-5 relative is far below the BF16 activations' resolution.  The
initial sweep still propagates the states.
"""

import ctypes
import sys
import time
from typing import Callable, Optional, Sequence, Union

import numpy as np

from pararealml_amd import _device as dev
from pararealml_amd import _native as nat
from pararealml_amd.initial_value_problem import InitialValueProblem
from pararealml_amd.operator import Operator, discretize_time_domain
from pararealml_amd.solution import DeviceSolution, Solution

TerminationCondition = Union[
    float, Sequence[float], Callable[[np.ndarray, np.ndarray], bool]
]


class PararealOperator(Operator):
    """A parallel-in-time solver based on the Parareal algorithm."""

    def __init__(
        self,
        f: Operator,
        g,
        termination_condition: TerminationCondition = None,
        max_iterations: int = sys.maxsize,
        *,
        n_slices: int = 1,
        output: str = "trajectory",
        monitor: Optional[Callable] = None,
        coarse_increments: bool = False,
    ):
        super().__init__(f.d_t, f.vertex_oriented)
        if n_slices < 1:
            raise ValueError("n_slices must be at least 1")
        if output not in ("trajectory", "endpoints"):
            raise ValueError("output must be 'trajectory' or 'endpoints'")
        self._f = f
        self._g = g
        self._termination_condition = termination_condition
        self._max_iterations = max_iterations
        self._n_slices = int(n_slices)
        self._output = output
        self._monitor = monitor
        self._coarse_increments = bool(coarse_increments)
        self.last_iterations: Optional[int] = None
        self.last_stats: dict = {}

    @property
    def n_slices(self) -> int:
        return self._n_slices

    # ------------------------------------------------------------ termination
    def _tolerances(self, y_dim: int) -> np.ndarray:
        tc = self._termination_condition
        if isinstance(tc, Sequence):
            if len(tc) != y_dim:
                raise ValueError(
                    f"length of update tolerances ({len(tc)}) must match number "
                    f"of y dimensions ({y_dim})"
                )
            return np.array(tc, dtype=float)
        return np.array([tc] * y_dim, dtype=float)

    # ------------------------------------------------------------------ solve
    def solve(self, ivp: InitialValueProblem, parallel_enabled: bool = True) -> Solution:
        if not parallel_enabled:
            return self._f.solve(ivp)
        import torch

        f, g = self._f, self._g
        n = self._n_slices
        t0, t1 = ivp.t_interval
        delta = (t1 - t0) / n
        if not np.isclose(delta, f.d_t * round(delta / f.d_t)):
            raise ValueError(
                f"fine operator time step size ({f.d_t}) must be a divisor of "
                f"sub-IVP time slice length ({delta})"
            )
        if not np.isclose(delta, g.d_t * round(delta / g.d_t)):
            raise ValueError(
                f"coarse operator time step size ({g.d_t}) must be a divisor of "
                f"sub-IVP time slice length ({delta})"
            )
        cp = ivp.constrained_problem
        tc = self._termination_condition
        if not callable(tc):
            tols = self._tolerances(cp.differential_equation.y_dimension)
        increments = self._coarse_increments
        if increments:
            _check_linear_homogeneous(cp)
            if getattr(g, "freeze", False):
                raise ValueError("a frozen correction is not linear in the state; use "
                                 "freeze=False with coarse_increments")
        f_steps = int(round(delta / f.d_t))
        g_steps = int(round(delta / g.d_t))
        borders = np.linspace(t0, t1, n + 1)

        stream = dev.solver_stream()
        stream.wait_stream(torch.cuda.current_stream())
        timings = {"fine_s": 0.0, "coarse_s": 0.0, "correction_s": 0.0}
        with torch.cuda.stream(stream):
            fine = f.slice_propagator(
                cp, n, f_steps, stream, record_trajectory=self._output == "trajectory",
                borders=borders,
            )
            coarse = g.slice_propagator(cp, n, g_steps, stream, borders=borders)
            problem = fine.problem
            elems = problem.elems
            plane = problem.plane
            n_fields = problem.n_fields
            lib = nat.device_lib()
            sp = ctypes.c_void_p(stream.cuda_stream)
            spatial = tuple(cp.y_vertices_shape[:-1])
            f64 = dict(dtype=torch.float64, device="cuda")

            y0 = ivp.initial_condition.discrete_y_0(True)
            u = torch.empty((n + 1, elems), **f64)
            u[0] = torch.from_numpy(problem.to_device_layout(y0).ravel()).to("cuda")
            g_end = torch.empty((n, elems), **f64)
            f_end = torch.empty((n, elems), **f64)
            corr = torch.empty((n, elems), **f64)
            inc = torch.empty((1, elems), **f64)  # U_new[j] - U_old[j]
            sumsq = torch.zeros((n, n_fields), **f64)
            reduce_work = torch.empty(nat.PML_REDUCE_SLOTS * n_fields, **f64)

            def sync_time(key, fn):
                stream.synchronize()
                start = time.perf_counter()
                fn()
                stream.synchronize()
                timings[key] += time.perf_counter() - start

            # A learned coarse propagator tests each slice for its fallback;
            # deferred, the tests cost one host synchronisation per sweep:
            # a sweep is re-run from the first flagged slice with that slice
            # computed by the fallback, as a test per slice would have done.
            deferred = (getattr(coarse, "supports_deferral", False)
                        and coarse.fallback is not None)
            if deferred:
                coarse.deferred = True

            def guarded(sweep_from, start, before_redo=None):
                sweep_from(start)
                if deferred:
                    while True:
                        jb = coarse.first_bad()
                        if jb is None:
                            break
                        coarse.force_fallback(jb)
                        if before_redo is not None:
                            before_redo(jb)
                        sweep_from(jb)
                    coarse.clear_forced()

            # initial coarse sweep
            def first_sweep(start):
                for j in range(start, n):
                    coarse.run(u[j : j + 1], j, j + 1, g_end[j : j + 1])
                    u[j + 1].copy_(g_end[j])

            sync_time("coarse_s", lambda: guarded(first_sweep, 0))

            iterations = 0
            norms_hist = []
            iter_wall = []
            for i in range(min(n, self._max_iterations)):
                iterations = i + 1
                sync_time("fine_s", lambda: fine.run(u[i:n], i, n, f_end[i:n]))

                def correct():
                    nat.check(
                        lib.pml_parareal_correction(
                            nat.PML_F64, f_end[i].data_ptr(), None, elems,
                            g_end[i].data_ptr(), corr[i].data_ptr(), elems, n - i, sp,
                        )
                    )

                if not increments:
                    sync_time("correction_s", correct)
                old = u[1:].clone() if callable(tc) else None
                prev = u.clone() if increments or deferred else None
                sumsq.zero_()

                def redo(jb):
                    # the update kernel adds to the norms and measures the
                    # change against u: restore both from slice jb on
                    u[jb + 1 :].copy_(prev[jb + 1 :])
                    sumsq[jb:].zero_()

                def sweep(start):
                    for j in range(start, n):
                        if increments:
                            # U[j+1] = G(U_new[j] - U_old[j]) + F(U_old[j])
                            if j > i:
                                nat.check(lib.pml_parareal_correction(
                                    nat.PML_F64, u[j].data_ptr(), None, elems,
                                    prev[j].data_ptr(), inc[0].data_ptr(), elems, 1, sp))
                                coarse.run(inc, j, j + 1, g_end[j : j + 1])
                            else:
                                g_end[j].zero_()  # U_new[i] == U_old[i]
                            src = f_end[j]
                        else:
                            if j > i:
                                coarse.run(u[j : j + 1], j, j + 1, g_end[j : j + 1])
                            src = corr[j]
                        nat.check(
                            lib.pml_parareal_update(
                                g_end[j].data_ptr(), src.data_ptr(),
                                u[j + 1].data_ptr(), elems, n_fields,
                                sumsq[j].data_ptr(), reduce_work.data_ptr(), sp,
                            )
                        )

                sync_time("coarse_s", lambda: guarded(sweep, i, redo))
                iter_wall.append(sum(timings.values()))
                if self._monitor is not None and self._monitor(i, u):
                    break
                if callable(tc):
                    layout = lambda t: problem.from_device_layout(  # noqa: E731
                        t.cpu().numpy().reshape(n, n_fields, problem.n0, problem.n1),
                        spatial,
                    )
                    if tc(layout(old), layout(u[1:])):
                        break
                else:
                    rms = np.sqrt(sumsq.cpu().numpy() / plane)
                    max_norms = rms.max(axis=0)
                    norms_hist.append(max_norms.tolist())
                    if np.all(max_norms < tols):
                        break

            self.last_iterations = iterations
            if self._output == "endpoints":
                dev_y = f_end + (u[1:] - f_end)
                y = dev.states_to_host(dev_y, problem, spatial)
                t = borders[1:]
                d_t_out = delta
            else:
                traj = fine.trajectory_f64()  # (steps, n, elems)
                shift = (u[1:] - traj[-1]).unsqueeze(0)
                dev_y = (traj + shift).permute(1, 0, 2).reshape(n * f_steps, elems)
                y = dev.states_to_host(dev_y, problem, spatial)
                t = discretize_time_domain(ivp.t_interval, f.d_t)[1:]
                d_t_out = f.d_t
        torch.cuda.current_stream().wait_stream(stream)
        self.last_stats = dict(
            timings, iterations=iterations, update_norms=norms_hist, iteration_wall_s=iter_wall
        )
        return DeviceSolution(ivp, t, y, dev_y, vertex_oriented=self._vertex_oriented,
                              d_t=d_t_out, field_major=True, copy=False)


_LINEAR_FAMILIES = ("diffusion", "convection_diffusion", "wave")


def _check_linear_homogeneous(cp) -> None:
    """The increment form needs G(a) - G(b) == G(a - b): a linear equation
    with homogeneous (zero) boundary values."""
    params = cp.differential_equation.device_parameters()
    if params is None or params[0] not in _LINEAR_FAMILIES:
        raise ValueError(
            "coarse_increments needs a linear equation (diffusion, convection-diffusion, "
            f"wave); got {type(cp.differential_equation).__name__}"
        )
    bc = dev.device_problem(cp).bc
    values = bc[~np.isnan(bc)]
    if values.size and np.any(values != 0.0):
        raise ValueError("coarse_increments needs homogeneous (zero) boundary values")
