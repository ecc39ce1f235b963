"""Device results on their way to the host: the channel-last copy and the
threaded download into pageable memory (``pml_download``), at sizes around
its 1 MiB pieces and its eight workers, on a stream with work queued, and
from several host threads at once."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PIECE = (1 << 20) // 8


@pytest.mark.parametrize("n", [1, PIECE - 1, PIECE, PIECE + 1, 7 * PIECE + 3, 8 * PIECE,
                               17 * PIECE + 5])
def test_download_equals_the_tensor(n):
    import torch

    from pararealml_amd import _device as dev
    from pararealml_amd import _native as nat

    print(f"case: download {n}", flush=True)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        t = torch.arange(n, dtype=torch.float64, device="cuda")
        for _ in range(50):  # queued work that the copy has to wait for
            t = t + 1.0
        got = dev.to_host(t)
    assert np.array_equal(got, np.arange(n) + 50.0)
    out = np.full(n + 2, -1.0)  # nothing beside the destination is written
    nat.check(nat.device_lib().pml_download(out.ctypes.data + 8, t.data_ptr(), 8 * n,
                                            stream.cuda_stream))
    assert out[0] == -1.0 and out[-1] == -1.0 and np.array_equal(out[1:-1], got)
    copy = dev.host_copy(got)
    assert np.array_equal(copy, got) and not np.shares_memory(copy, got)


def test_concurrent_downloads():
    import torch

    from pararealml_amd import _device as dev
    from pararealml_amd import _native as nat

    print("case: concurrent downloads", flush=True)
    sources = [torch.full((5 * PIECE + k,), float(k), dtype=torch.float64, device="cuda")
               for k in range(4)]
    torch.cuda.synchronize()
    results = [None] * 4

    def fetch(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            results[k] = dev.to_host(sources[k])

    threads = [threading.Thread(target=fetch, args=(k,)) for k in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for k, r in enumerate(results):
        assert r.shape == (5 * PIECE + k,) and np.all(r == float(k))
    nat.check(nat.device_lib().pml_graph_cache_clear())  # gives the staging back
    assert np.all(dev.to_host(sources[3]) == 3.0)


@pytest.mark.parametrize("fields", [1, 2, 3, 4])
@pytest.mark.parametrize("plane,states", [(1, 5), (255, 3), (256, 1), (1025, 7)])
def test_channel_last(fields, plane, states):
    import torch

    from pararealml_amd import _native as nat

    print(f"case: channel last {fields} {plane} {states}", flush=True)
    x = torch.rand(states, fields, plane, dtype=torch.float64, device="cuda")
    out = torch.empty(states, plane, fields, dtype=torch.float64, device="cuda")
    nat.check(nat.device_lib().pml_channel_last(
        x.data_ptr(), out.data_ptr(), fields, plane, states,
        torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, x.movedim(1, 2))
