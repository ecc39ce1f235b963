"""Downloads behind work queued on each kind of stream, the one that belongs to
the calling thread among them: the copying threads have another of that name."""

import ctypes

import numpy as np
import pytest

import pararealml_amd as pml

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread


@pytest.mark.parametrize("kind", ["default", "own", "per thread"])
def test_downloads_wait_for_the_queued_work(kind):
    import torch

    from pararealml_amd import _device as dev
    from pararealml_amd import _native as nat

    print(f"case: download behind work on a {kind} stream", flush=True)
    n = 2000
    mesh = pml.Mesh([(0.0, 1.0)] * 2, [1.0 / (n - 1)] * 2)
    bc = pml.DirichletBoundaryCondition(lambda x, t: np.zeros((len(x), 1)), is_static=True)
    cp = pml.ConstrainedProblem(pml.DiffusionEquation(2, 0.5), mesh, [(bc, bc)] * 2)
    b = dev.FDMBatch([dev.device_problem(cp)], [0], "float64", nat.PML_INT_RK4)
    b.load_host([np.random.RandomState(0).uniform(-1.0, 1.0, (n, n, 1))])
    own = torch.cuda.Stream()
    torch.cuda.synchronize()
    stream = ctypes.c_void_p(
        {"default": 0, "own": own.cuda_stream, "per thread": PER_THREAD}[kind])
    nat.check(b.lib.pml_fdm_solve(
        b.eq_id, b._params, len(b.params), b.integrator, b.prec, b.ndim, b.grids, 1,
        b.bc.data_ptr(), b.hi.data_ptr(), None, b.work_hi.data_ptr(), None, b.total, 1e-8, 400,
        None, None, 0, 0, 0, stream))  # tens of milliseconds
    got = np.empty(b.total)
    nat.check(b.lib.pml_download(got.ctypes.data, b.hi.data_ptr(), got.nbytes, stream))
    torch.cuda.synchronize()
    assert np.array_equal(got, b.hi.cpu().numpy())
