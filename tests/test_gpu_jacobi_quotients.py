"""The divisions of the Jacobi iteration against NumPy's: equal to the bit for
one sweep (``pml_jacobi_sweep``), for the loop in one workgroup and for the
loop of two launches a sweep (``pml_jacobi_solve``), for values of ordinary
size, for values whose products with a reciprocal leave the range of exact
residuals, for zeros of both signs, and with infinities among the values."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# plates and a box in one workgroup (two, and up to 18 vertices a thread), and
# a plate and a box above its limits
SHAPES = [(40, 44), (64, 100), (12, 11, 10), (150, 160), (24, 23, 22)]
SPACING = [0.1, 0.125, 0.2]


def _values(kind, shape, dtype):
    rng = np.random.RandomState(len(kind) + sum(shape))
    y = rng.uniform(-1.0, 1.0, shape)
    if kind == "tiny":
        # powers of two down to the subnormal numbers
        low, high = (-125, -108) if dtype == np.float32 else (-1021, -960)
        y = np.sign(y) * 2.0 ** (low + (high - low) * np.abs(y))
    elif kind == "huge":
        y = y * (2.0**122 if dtype == np.float32 else 2.0**1018)
    elif kind == "infinite":
        y[tuple(rng.randint(0, n, 9) for n in shape)] = np.inf
    elif kind == "zeros":
        y = np.where(rng.uniform(size=shape) < 0.7, np.copysign(0.0, y), y)
    return y.astype(dtype)


def _sweep(y, lap, fixed):
    """numerical_differentiator.py:1097-1186: neighbours beyond the grid are
    0, vertices with a fixed value keep it."""
    t = y.dtype.type
    acc, coef = np.zeros_like(y), 0.0
    with np.errstate(all="ignore"):
        for axis, d in enumerate(SPACING[:y.ndim]):
            pad = [(1, 1) if a == axis else (0, 0) for a in range(y.ndim)]
            p = np.pad(y, pad)
            n = y.shape[axis]
            prev, nxt = p.take(range(n), axis), p.take(range(2, n + 2), axis)
            acc = acc + (prev + nxt) / t(d * d)
            coef += 2.0 / (d * d)
        new = (acc - lap) / t(coef)
    return np.where(np.isnan(fixed), new, fixed.astype(y.dtype))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["ordinary", "tiny", "huge", "zeros", "infinite"])
@pytest.mark.parametrize("shape", SHAPES)
def test_quotients_of_the_jacobi_sweeps(shape, kind, dtype):
    import torch

    from pararealml_amd import _native as nat

    print(f"case: jacobi quotients {shape} {kind} {dtype.__name__}", flush=True)
    prec = nat.PML_F64 if dtype == np.float64 else nat.PML_F32
    y = _values(kind, shape, dtype)
    lap = _values(kind, shape[::-1], dtype).reshape(shape)
    lap[~np.isfinite(lap)] = 0.0
    fixed = np.full(shape, np.nan)
    if len(shape) == 2:  # all edges, or the plate of 64 x 100 is no longer in one workgroup
        fixed[-1] = fixed[:, 0] = fixed[:, -1] = 0.25
    fixed[0] = 0.25
    y[~np.isnan(fixed)] = 0.25
    want = _sweep(y, lap, fixed)
    twice = _sweep(want, lap, fixed)
    dims = list(shape) + [1] * (3 - len(shape))
    c_shape = (ctypes.c_int64 * 3)(*dims)
    dx = (ctypes.c_double * 3)(*(SPACING[:len(shape)] + [1.0] * (3 - len(shape))))
    none = (ctypes.c_void_p * 3)()
    lib, st = nat.device_lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    yd, ld, fd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (y, lap, fixed))
    out, spare = torch.empty_like(yd), torch.empty_like(yd)
    norm = torch.zeros(1, dtype=torch.float64, device="cuda")
    work = torch.zeros(nat.PML_REDUCE_SLOTS, dtype=torch.float64, device="cuda")
    # the loop of two launches leaves its partial sums here
    state = torch.full((nat.PML_JACOBI_STATE_BYTES // 8,), -1.0, dtype=torch.float64,
                       device="cuda")
    nat.check(lib.pml_jacobi_sweep(prec, yd.data_ptr(), out.data_ptr(), ld.data_ptr(), c_shape, 1,
                                   dx, none, none, fd.data_ptr(), norm.data_ptr(),
                                   work.data_ptr(), st))
    # array_equal takes -0 for 0: the sign bits are compared beside it
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    assert np.array_equal(np.signbit(out.cpu().numpy()) & (want == 0),
                          np.signbit(want) & (want == 0))
    sweeps, diff = ctypes.c_int64(0), ctypes.c_double(0.0)
    cur = yd.clone()
    nat.check(lib.pml_jacobi_solve(prec, cur.data_ptr(), spare.data_ptr(), ld.data_ptr(), c_shape,
                                   1, dx, none, none, fd.data_ptr(), 0.0, 2, 64,
                                   state.data_ptr(), ctypes.byref(sweeps), ctypes.byref(diff), st))
    assert bool((state[4:] == -1.0).all()) == (shape in SHAPES[:3])
    np.testing.assert_array_equal(cur.cpu().numpy(), twice)
    assert np.array_equal(np.signbit(cur.cpu().numpy()) & (twice == 0),
                          np.signbit(twice) & (twice == 0))
