"""Results for the host from tensors of any layout, and the device memory that
their transposition may take."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_strided_tensors_reach_the_host_as_they_are():
    import torch

    from pararealml_amd import _device as dev

    print("case: strided results", flush=True)
    base = torch.rand(1024, 768, dtype=torch.float64, device="cuda")  # above the threaded size
    for view in (base.t(), base[:, ::2], base[3:, 5:], base.view(32, 32, 768).permute(2, 0, 1)):
        assert np.array_equal(dev.to_host(view), view.cpu().numpy())


class _Problem:
    n_fields, n0, n1 = 3, 40, 50
    plane = 2000


def _want(states):
    flat = states.cpu().numpy().reshape(-1, 3, 40, 50)
    return np.moveaxis(flat, 1, -1)


def test_strided_states_are_transposed_as_they_are():
    import torch

    from pararealml_amd import _device as dev

    print("case: strided states", flush=True)
    base = torch.rand(6000, 120, dtype=torch.float64, device="cuda")
    for states in (base.t(), base.t()[::2]):
        assert np.array_equal(dev.states_to_host(states, _Problem, (40, 50)), _want(states))


@pytest.mark.parametrize("n", [1, 21, 22, 64])
def test_transposed_states_need_bounded_device_memory(n, monkeypatch):
    import torch

    from pararealml_amd import _device as dev

    print(f"case: bounded transposition {n}", flush=True)
    limit = 1 << 20  # 21 states of 48 kB
    monkeypatch.setattr(dev, "_TRANSPOSED_BYTES", limit, raising=False)
    states = torch.rand(n + 21, 6000, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = dev.states_to_host(states, _Problem, (40, 50))
    assert torch.cuda.max_memory_allocated() - before <= limit
    assert np.array_equal(got, _want(states))
    # one state beyond the limit goes by itself
    monkeypatch.setattr(dev, "_TRANSPOSED_BYTES", 1, raising=False)
    assert np.array_equal(dev.states_to_host(states, _Problem, (40, 50)), _want(states))
