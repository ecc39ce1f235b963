// How a run of the many-step kernel is cut into launches (host only).
#pragma once

#include <algorithm>
#include <cstdint>

namespace pml {

// The launch that begins after `done` of n_steps steps: its steps, the index
// of the next snapshot, the steps to it, and those between further ones.  A
// launch has at most `most` steps, and its counters 31 bits: steps beyond
// those are out of its reach and may stand at any value that is.
struct DeepLaunch {
  int steps;
  int64_t snap_idx;
  int until, every;
};

// snapshot_every 0: no snapshots.
inline DeepLaunch deep_launch(int most, int64_t n_steps, int64_t done, int64_t snapshot_every) {
  constexpr int64_t kBeyond = int64_t{1} << 30;
  DeepLaunch l{static_cast<int>(std::min<int64_t>(most, n_steps - done)), 0,
               static_cast<int>(kBeyond), static_cast<int>(kBeyond)};
  if (snapshot_every > 0) {
    l.snap_idx = done / snapshot_every;
    l.until = static_cast<int>(std::min(snapshot_every - done % snapshot_every, kBeyond));
    l.every = static_cast<int>(std::min(snapshot_every, kBeyond));
  }
  return l;
}

}  // namespace pml
