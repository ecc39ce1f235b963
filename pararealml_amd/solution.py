"""Solutions of initial value problems.

Semantics follow pararealml/solution.py:22-258 and 329-336 (constructor
validation and copying, interpolation, orientation conversion, and the
time-matched differences).  Plotting (solution.py:260-326) is presentation
and is not part of this package.
"""

from __future__ import annotations

from typing import List, NamedTuple, Optional, Sequence

import numpy as np
from scipy.interpolate import interpn

from pararealml_amd.constraint import apply_constraints_along_last_axis
from pararealml_amd.initial_value_problem import InitialValueProblem


class Solution:
    """A discrete solution: time coordinates and ``(n_t, *y_shape)`` values."""

    def __init__(
        self,
        ivp: InitialValueProblem,
        t_coordinates: np.ndarray,
        discrete_y: np.ndarray,
        vertex_oriented: Optional[bool] = None,
        d_t: Optional[float] = None,
        *,
        copy: bool = True,
    ):
        if t_coordinates.ndim != 1:
            raise ValueError(
                f"number of t coordinate dimensions ({t_coordinates.ndim}) "
                "must be 1"
            )
        if len(t_coordinates) == 0:
            raise ValueError("length of t coordinates must be greater than 0")
        cp = ivp.constrained_problem
        if cp.differential_equation.x_dimension and vertex_oriented is None:
            raise ValueError(
                "vertex orientation must be defined for solutions to PDEs"
            )
        y_shape = cp.y_shape(vertex_oriented)
        if discrete_y.shape != (len(t_coordinates),) + y_shape:
            raise ValueError(
                "expected solution shape to be "
                f"{(len(t_coordinates),) + y_shape} but got {discrete_y.shape}"
            )
        self._ivp = ivp
        self._t_coordinates = np.array(t_coordinates, copy=True)
        # copy=False: the caller hands over an array that nobody else holds
        self._discrete_y = np.array(discrete_y, copy=True) if copy else discrete_y
        self._vertex_oriented = vertex_oriented
        self._t_coordinates.setflags(write=False)
        if d_t is None:
            d_t = (
                0.0
                if len(t_coordinates) == 1
                else t_coordinates[1] - t_coordinates[0]
            )
        self._d_t = d_t

    @property
    def initial_value_problem(self) -> InitialValueProblem:
        return self._ivp

    @property
    def vertex_oriented(self) -> Optional[bool]:
        return self._vertex_oriented

    @property
    def d_t(self) -> float:
        return self._d_t

    @property
    def t_coordinates(self) -> np.ndarray:
        return self._t_coordinates

    def y(
        self, x: Optional[np.ndarray] = None, interpolation_method: str = "linear"
    ) -> np.ndarray:
        """Values at arbitrary spatial points for every time step
        (pararealml/solution.py:114-145)."""
        cp = self._ivp.constrained_problem
        diff_eq = cp.differential_equation
        if not diff_eq.x_dimension:
            return self._values_copy()
        values = interpn(
            cp.mesh.axis_coordinates(self._vertex_oriented),
            np.moveaxis(self._discrete_y, 0, -2),
            x,
            method=interpolation_method,
            bounds_error=False,
            fill_value=None,
        )
        values = np.moveaxis(values, -2, 0)
        values = values.reshape(
            (len(self._t_coordinates),) + x.shape[:-1] + (diff_eq.y_dimension,)
        )
        return np.ascontiguousarray(values)

    def _values_copy(self) -> np.ndarray:
        return np.copy(self._discrete_y)

    def discrete_y(
        self,
        vertex_oriented: Optional[bool] = None,
        interpolation_method: str = "linear",
    ) -> np.ndarray:
        """The solution on vertices or cell centres
        (pararealml/solution.py:147-180)."""
        if vertex_oriented is None:
            vertex_oriented = self._vertex_oriented
        cp = self._ivp.constrained_problem
        if (
            not cp.differential_equation.x_dimension
            or self._vertex_oriented == vertex_oriented
        ):
            return self._values_copy()
        x = cp.mesh.all_index_coordinates(vertex_oriented)
        values = self.y(x, interpolation_method)
        if vertex_oriented:
            apply_constraints_along_last_axis(cp.static_y_vertex_constraints, values)
        return values

    def diff(self, solutions: Sequence["Solution"], atol: float = 1e-8) -> "Diffs":
        """Differences to other solutions at matching time points
        (pararealml/solution.py:182-258)."""
        if len(solutions) == 0:
            raise ValueError("length of solutions must be greater than 0")
        all_t = [self._t_coordinates] + [s.t_coordinates for s in solutions]
        all_dt = [self._d_t] + [s.d_t for s in solutions]
        others = [s.discrete_y(self._vertex_oriented) for s in solutions]
        matching, indices = _matching_indices(all_t, all_dt, atol)
        diffs: List[List[np.ndarray]] = [[] for _ in solutions]
        for i in range(len(matching)):
            for j, other in enumerate(others):
                diffs[j].append(other[indices[j + 1][i]] - self._discrete_y[indices[0][i]])
        return Diffs(np.array(matching), [np.array(d) for d in diffs])


def _matching_indices(all_t, all_dt, atol: float):
    """The time points of the solution with the fewest that every other
    solution matches within ``atol`` at index ``round((t - t_0) / d_t)``,
    and the matched snapshot index per solution (solution.py:203-240)."""
    shortest = int(np.argmin([len(t) for t in all_t]))
    matching: List[float] = []
    indices: List[List[int]] = [[] for _ in all_t]
    for i, t in enumerate(all_t[shortest]):
        found = []
        for j, t_j in enumerate(all_t):
            if j == shortest:
                found.append(i)
                continue
            k = int(round((t - t_j[0]) / all_dt[j]))
            if 0 <= k < len(t_j) and np.isclose(t, t_j[k], atol=atol, rtol=0.0):
                found.append(k)
            else:
                found = None
                break
        if found is None:
            continue
        matching.append(t)
        for j, k in enumerate(found):
            indices[j].append(k)
    return matching, indices


# Interpolation methods evaluated on the device: SciPy's "slinear" is its
# spline form of "linear" and gives the same values up to rounding.
_DEVICE_METHODS = {"linear": 0, "slinear": 0, "nearest": 1}


class DeviceSolution(Solution):
    """A solution computed on the GPU that keeps its FP64 snapshots in device
    memory beside the host copy the reference's API hands out.

    ``y`` and the orientation change of ``discrete_y`` interpolate on the
    device (``pml_interp_regular``: SciPy's ``interpn`` semantics, FP64
    results equal to SciPy's), ``diff`` subtracts the matched snapshots on
    the device (``pml_snapshot_diff``); both return host arrays, as the
    reference (solution.py:114-258) does, and ``y_device`` / ``diff_device``
    return device tensors.  On the device, interpolation covers "linear"
    (also for "slinear") and "nearest"; other methods raise
    ``NotImplementedError``.

    ``device_y`` holds the snapshots channel-last, ``(n_t, *y_shape)``, or,
    with ``field_major``, ``(n_t, y_dim, *grid)`` -- the layout of the fused
    solvers, read in place.
    """

    def __init__(
        self,
        ivp: InitialValueProblem,
        t_coordinates: np.ndarray,
        discrete_y: np.ndarray,
        device_y,
        vertex_oriented: Optional[bool] = None,
        d_t: Optional[float] = None,
        field_major: bool = False,
        *,
        copy: bool = True,
    ):
        super().__init__(ivp, t_coordinates, discrete_y, vertex_oriented, d_t, copy=copy)
        import torch

        if not isinstance(device_y, torch.Tensor) or not device_y.is_cuda:
            raise ValueError("device_y must be a tensor in GPU memory")
        if device_y.numel() != self._discrete_y.size:
            raise ValueError(
                f"device snapshots hold {device_y.numel()} values, expected "
                f"{self._discrete_y.size}"
            )
        self._device_y = device_y.to(torch.float64).contiguous().view(-1)
        self._field_major = bool(field_major) and bool(
            ivp.constrained_problem.differential_equation.x_dimension
        )
        self._coords = None
        self._time_inner = None

    def _values_copy(self) -> np.ndarray:
        from pararealml_amd import _device as dev

        return dev.host_copy(self._discrete_y)

    @property
    def device_y(self):
        """The device snapshots (flat FP64 tensor in the layout above)."""
        return self._device_y

    @property
    def field_major(self) -> bool:
        return self._field_major

    def _layout(self):
        cp = self._ivp.constrained_problem
        y_shape = cp.y_shape(self._vertex_oriented)
        c = cp.differential_equation.y_dimension
        points = int(np.prod(y_shape[:-1])) if len(y_shape) > 1 else 1
        return points, c

    def y_device(self, x, interpolation_method: str = "linear"):
        """``y(x)`` as a device tensor ``(n_t, *x.shape[:-1], y_dim)``.

        When the output is at least as large as the snapshot stack (and
        there are 16 snapshots or more), the stack is first copied once
        into the time-inner layout (kept with the solution), in which every
        corner read of a query point is one contiguous run of its
        snapshots; smaller queries read the stack in place.  Both paths
        give identical values."""
        return self._interp(x, interpolation_method, None)

    def _time_inner_stack(self):
        import torch

        from pararealml_amd import _native as nat

        if self._time_inner is None:
            points, c = self._layout()
            n_t = len(self._t_coordinates)
            vt = torch.empty_like(self._device_y)
            stream = torch.cuda.current_stream(self._device_y.device)
            self._device_y.record_stream(stream)
            layout = (nat.PML_LAYOUT_FIELD_MAJOR if self._field_major
                      else nat.PML_LAYOUT_CHANNEL_LAST)
            nat.check(nat.device_lib().pml_snapshots_time_inner(
                nat.PML_F64, layout, self._device_y.data_ptr(), n_t, points, c,
                vt.data_ptr(), stream.cuda_stream))
            self._time_inner = vt
        return self._time_inner

    def _interp(self, x, interpolation_method: str, time_inner: Optional[bool]):
        import ctypes

        import torch

        from pararealml_amd import _native as nat

        cp = self._ivp.constrained_problem
        if not cp.differential_equation.x_dimension:
            return self._device_y.view(self._discrete_y.shape).clone()
        method = _DEVICE_METHODS.get(interpolation_method)
        if method is None:
            raise NotImplementedError(
                f"interpolation method {interpolation_method!r} is not evaluated on the "
                "device (linear, slinear and nearest are)"
            )
        lib = nat.device_lib()
        axes = cp.mesh.axis_coordinates(self._vertex_oriented)
        d = len(axes)
        device = self._device_y.device
        xt = torch.as_tensor(x, dtype=torch.float64).to(device)
        if xt.ndim == 0 or xt.shape[-1] != d:
            got = xt.shape[-1] if xt.ndim else 0
            raise ValueError(
                f"The requested sample points xi have dimension {got} but this "
                f"RegularGridInterpolator has dimension {d}"
            )
        pts = xt.reshape(-1, d).contiguous()
        if self._coords is None:
            flat = np.concatenate([np.asarray(a, dtype=np.float64) for a in axes])
            self._coords = torch.from_numpy(flat).to(device)
        shape = (ctypes.c_int64 * d)(*[len(a) for a in axes])
        n_t = len(self._t_coordinates)
        points, c = self._layout()
        if time_inner is None:
            time_inner = n_t >= 16 and pts.shape[0] >= points
        if time_inner:
            values, layout = self._time_inner_stack(), nat.PML_LAYOUT_TIME_INNER
        elif self._field_major:
            values, layout = self._device_y, nat.PML_LAYOUT_FIELD_MAJOR
        else:
            values, layout = self._device_y, nat.PML_LAYOUT_CHANNEL_LAST
        out = torch.empty((n_t, pts.shape[0], c), dtype=torch.float64, device=device)
        stream = torch.cuda.current_stream(device)
        values.record_stream(stream)
        nat.check(
            lib.pml_interp_regular(
                nat.PML_F64, method, layout, values.data_ptr(), n_t, d, shape, c,
                self._coords.data_ptr(), pts.data_ptr(), pts.shape[0], out.data_ptr(),
                stream.cuda_stream,
            )
        )
        return out.view((n_t,) + tuple(xt.shape[:-1]) + (c,))

    def y(
        self, x: Optional[np.ndarray] = None, interpolation_method: str = "linear"
    ) -> np.ndarray:
        """Values at arbitrary spatial points for every time step
        (pararealml/solution.py:114-145), interpolated on the device."""
        if not self._ivp.constrained_problem.differential_equation.x_dimension:
            return self._values_copy()
        return np.ascontiguousarray(self.y_device(x, interpolation_method).cpu().numpy())

    def _device_stack(self, other: Solution):
        """``other``'s snapshots on the device in this solution's layout and
        orientation."""
        import torch

        if (
            isinstance(other, DeviceSolution)
            and other._vertex_oriented == self._vertex_oriented
            and other._field_major == self._field_major
        ):
            return other._device_y, len(other.t_coordinates)
        host = other.discrete_y(self._vertex_oriented)
        if self._field_major:
            host = np.moveaxis(host, -1, 1)
        dev_stack = torch.from_numpy(np.ascontiguousarray(host, dtype=np.float64))
        return dev_stack.to(self._device_y.device).view(-1), len(other.t_coordinates)

    def diff_device(self, solutions: Sequence[Solution], atol: float = 1e-8):
        """``diff`` with device results: (matched time points as a host
        array, [device tensor (n_matched, *y_shape) per solution])."""
        import torch

        from pararealml_amd import _native as nat

        if len(solutions) == 0:
            raise ValueError("length of solutions must be greater than 0")
        lib = nat.device_lib()
        all_t = [self._t_coordinates] + [s.t_coordinates for s in solutions]
        all_dt = [self._d_t] + [s.d_t for s in solutions]
        matching, indices = _matching_indices(all_t, all_dt, atol)
        points, c = self._layout()
        y_shape = self._discrete_y.shape[1:]
        device = self._device_y.device
        stream = torch.cuda.current_stream(device)
        self._device_y.record_stream(stream)
        n_a = len(self._t_coordinates)
        ia = torch.tensor(indices[0], dtype=torch.int64).to(device)
        outs = []
        for j, other in enumerate(solutions):
            other_cp = other.initial_value_problem.constrained_problem
            if tuple(other_cp.y_shape(self._vertex_oriented)) != tuple(y_shape):
                raise ValueError("solutions of different shapes cannot be compared")
            stack, n_b = self._device_stack(other)
            stack.record_stream(stream)
            ib = torch.tensor(indices[j + 1], dtype=torch.int64).to(device)
            out = torch.empty((len(matching),) + y_shape, dtype=torch.float64, device=device)
            nat.check(
                lib.pml_snapshot_diff(
                    nat.PML_F64, int(self._field_major), self._device_y.data_ptr(),
                    ia.data_ptr(), n_a, stack.data_ptr(), ib.data_ptr(), n_b,
                    out.data_ptr(), len(matching), points, c, stream.cuda_stream,
                )
            )
            outs.append(out)
        return np.array(matching), outs

    def diff(self, solutions: Sequence[Solution], atol: float = 1e-8) -> "Diffs":
        """Differences to other solutions at matching time points
        (pararealml/solution.py:182-258), subtracted on the device."""
        matching, outs = self.diff_device(solutions, atol)
        if len(matching) == 0:
            return Diffs(matching, [np.array([]) for _ in outs])
        return Diffs(matching, [o.cpu().numpy() for o in outs])


class Diffs(NamedTuple):
    """pararealml/solution.py:329-336."""

    matching_time_points: np.ndarray
    differences: Sequence[np.ndarray]
