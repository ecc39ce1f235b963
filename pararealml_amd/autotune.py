"""Tile-shape autotuner for the fused stepping kernels.

For an (equation, integrator, precision, grid-size class) key it times every
kernel variant ``libpml.so`` offers for that combination (tile height, fused
steps per launch, workgroup size -- ``pml_fdm_configs`` /
``pml_fdm_config_name``) and, where it has a plan for the batch, the many-step
kernel on the live device, on a scratch batch of the caller's shape, and keeps
the fastest.  Results persist as JSON in
``$PML_AUTOTUNE_CACHE`` (default ``~/.cache/pararealml_amd/autotune.json``)
and are reused by ``FDMOperator`` when it is not given a ``tile_config``.
The cache stores the variant's *name*; a lookup resolves it against the
variants the loaded library offers, so an entry written by another build
(pruned or reordered variants) falls back to the default variant instead
of selecting a wrong or out-of-range one.  " > many-step" or " < many-step"
after the name says that the many-step kernel was timed too and took less or
more time than the variant; it stays off only in the second case.
"""

import json
import os
import threading
from pathlib import Path
from typing import Dict, List, Optional, Sequence

MANY_STEP = "many-step"

_lock = threading.Lock()
_cache: Optional[Dict[str, str]] = None


def _cache_path() -> Path:
    env = os.environ.get("PML_AUTOTUNE_CACHE")
    if env:
        return Path(env)
    return Path.home() / ".cache" / "pararealml_amd" / "autotune.json"


def _load() -> Dict[str, str]:
    global _cache
    if _cache is None:
        path = _cache_path()
        try:
            raw = json.loads(path.read_text())
            # entries that are not variant names (e.g. bare indices) are stale
            _cache = {k: v for k, v in raw.items() if isinstance(v, str)}
        except (OSError, ValueError, AttributeError):
            _cache = {}
    return _cache


def variant_names(eq_id: int, integrator: int, prec: int) -> List[str]:
    """The kernel variants the loaded library offers, in index order."""
    from pararealml_amd import _native as nat

    lib = nat.load_library()
    return [
        lib.pml_fdm_config_name(eq_id, integrator, prec, i).decode()
        for i in range(lib.pml_fdm_configs(eq_id, integrator, prec))
    ]


def _size_class(cells: int) -> str:
    for bound, name in ((1 << 14, "xs"), (1 << 17, "s"), (1 << 20, "m"), (1 << 23, "l")):
        if cells <= bound:
            return name
    return "xl"


def key_for(problem, integrator: int, precision: str, cells: Optional[int] = None) -> str:
    cells = problem.plane if cells is None else cells
    return f"{problem.eq_name}/{integrator}/{precision}/{problem.ndim}d/{_size_class(cells)}"


def lookup(problem, integrator: int, precision: str, cells: Optional[int] = None,
           names: Optional[Sequence[str]] = None) -> int:
    """Index of the tuned variant for this key among ``names`` (default: the
    loaded library's variants), or 0 (the default variant) when nothing is
    recorded or the recorded name is not offered."""
    with _lock:
        name = _load().get(key_for(problem, integrator, precision, cells))
    if name is None:
        return 0
    if names is None:
        names = _offered(problem, integrator, precision)
    try:
        return list(names).index(name.split(" ")[0])
    except ValueError:
        return 0


def _offered(problem, integrator: int, precision: str) -> List[str]:
    from pararealml_amd import _device as dev
    from pararealml_amd import _native as nat

    return variant_names(nat.PML_EQ[problem.eq_name], integrator, dev.precision_id(precision))


def many_step(problem, integrator: int, precision: str, cells: Optional[int] = None) -> bool:
    """Whether batches of this key may run the many-step kernel: unless a
    tuning run recorded a variant this library offers as the faster one."""
    with _lock:
        name = _load().get(key_for(problem, integrator, precision, cells), "")
    variant, _, timed = name.partition(" ")
    return timed != "< " + MANY_STEP or variant not in _offered(problem, integrator, precision)


def tune(batch, d_t: float, n_steps: int = 64, repeats: int = 3, store: bool = True):
    """Times every variant and the many-step kernel on ``batch`` (an
    ``FDMBatch``; its state is advanced and therefore clobbered) and records
    the fastest.  Returns ``(best_config, {config_name: seconds_per_step})``:
    the fastest variant, beside which ``"many-step"`` may be faster yet."""
    import ctypes

    import torch

    from pararealml_amd import _native as nat

    lib = batch.lib
    names = variant_names(batch.eq_id, batch.integrator, batch.prec)
    plan = (ctypes.c_int * 4)()
    nat.check(lib.pml_fdm_auto_plan(batch.eq_id, batch.integrator, batch.prec, batch.ndim,
                                    batch.grids, len(batch.grid_problem), int(n_steps), plan))
    candidates = [(name, dict(tile_config=cfg)) for cfg, name in enumerate(names)]
    if plan[3]:
        candidates.append((MANY_STEP, dict(auto=True)))
    timings = {}
    for name, choice in candidates:
        batch.advance(d_t, 8, **choice)  # warm-up
        torch.cuda.synchronize()
        start = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        ts = []
        for _ in range(repeats):
            start.record(batch.stream)
            batch.advance(d_t, n_steps, use_graph=True, **choice)
            end.record(batch.stream)
            end.synchronize()
            ts.append(start.elapsed_time(end) / 1e3 / n_steps)
        timings[name] = min(ts)
    best = min(range(len(names)), key=lambda cfg: timings[names[cfg]])
    if store:
        cells = sum(batch.problems[i].plane for i in batch.grid_problem)
        key = key_for(batch.problems[0], batch.integrator, batch.precision, cells)
        entry = names[best]
        if MANY_STEP in timings:
            entry += (" > " if timings[MANY_STEP] < timings[entry] else " < ") + MANY_STEP
        with _lock:
            data = _load()
            data[key] = entry
            path = _cache_path()
            try:
                path.parent.mkdir(parents=True, exist_ok=True)
                path.write_text(json.dumps(data, indent=1, sort_keys=True))
            except OSError:
                pass
    return best, timings
