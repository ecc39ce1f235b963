"""How the many-step kernel's launches count the steps to the next snapshot
(``csrc/pml_launches.h``, compiled for the host): runs and intervals beyond
2^30 steps, which a launch's own counters would overflow on, and the snapshots
that all launches of a run write together."""

import ctypes
import subprocess

import pytest

from pararealml_amd.build import CSRC

SOURCE = """
#include "pml_launches.h"
extern "C" void launch(int most, int64_t n_steps, int64_t done, int64_t every, int64_t *out) {
  const pml::DeepLaunch l = pml::deep_launch(most, n_steps, done, every);
  out[0] = l.steps; out[1] = l.snap_idx; out[2] = l.until; out[3] = l.every;
}
"""


@pytest.fixture(scope="module")
def launch(tmp_path_factory):
    where = tmp_path_factory.mktemp("launches")
    (where / "launch.cpp").write_text(SOURCE)
    lib = where / "launch.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(lib),
                    str(where / "launch.cpp")], check=True)
    fn = ctypes.CDLL(str(lib)).launch
    fn.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.POINTER(ctypes.c_int64)]

    def call(*args):
        out = (ctypes.c_int64 * 4)()
        fn(*args, out)
        return tuple(out)

    return call


def _written(launch, most, n_steps, first, last, every):
    """(step, index) of the snapshots that the launches from step `first` on,
    up to step `last`, write: the kernel's counting."""
    done, seen = first, []
    while done < last:
        steps, snap, until, again = launch(most, n_steps, done, every)
        assert 0 < steps <= most and 0 < until < 2**31 and 0 < again < 2**31
        for step in range(done, done + steps):
            until -= 1
            if until == 0:
                seen.append((step + 1, snap))
                snap += 1
                until = again
        done += steps
    return seen


@pytest.mark.parametrize("most", [1, 7, 2048])
@pytest.mark.parametrize("every", [1, 3, 7, 100])
def test_snapshots_of_a_run(launch, most, every):
    assert _written(launch, most, 500, 0, 500, every) == [
        (s, s // every - 1) for s in range(1, 501) if s % every == 0]


def test_runs_without_snapshots_write_none(launch):
    for first in (0, 2**30 - 2048, 2**31 - 5000, 2**40):
        assert _written(launch, 2048, 2**41, first, first + 6000, 0) == []


@pytest.mark.parametrize("every", [2**30 + 1, 2**31, 2**33 + 7])
def test_intervals_beyond_the_counters(launch, every):
    for k in (1, 2, 5):
        first = k * every - 3000
        assert _written(launch, 2048, 2**41, first, first + 4000, every) == [(k * every, k - 1)]
