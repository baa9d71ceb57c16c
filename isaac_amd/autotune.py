"""Launch-schedule autotuner.

Times the march kernel of a visualization under each candidate schedule
(include/isaac_hip.h, "tuning": the tile order over the XCDs and, in the combined form,
the workgroup size: one wave or 4) on the caller's own frames and keeps the fastest.
Results do not depend on the schedule, only speed does; choices are cached per workload
key.
"""
from __future__ import annotations

import itertools
from typing import Dict, Sequence, Tuple

import numpy as np

_CACHE: Dict[Tuple, Dict[str, int]] = {}

CANDIDATES = {
    "march_tiles": (0, 4, 8),
    "march_threads": (64, 256),
}


def _key(vis) -> Tuple:
    return (vis.framebuffer_size, vis.local_size, len(vis.volume_sources), len(vis.particle_sources),
            bool(vis.interpolation), vis.render_form)


def _apply(vis, choice: Dict[str, int]) -> None:
    vis.set_tuning(vis.TUNE_MARCH_TILES, choice["march_tiles"])
    # (a choice for the brick form, whose march has one workgroup size, has none: the one that the
    # context keeps is the combined form's)
    if "march_threads" in choice:
        vis.set_tuning(vis.TUNE_MARCH_THREADS, choice["march_threads"])


def tune_march(vis, poses: Sequence, frames: int = 4, use_cache: bool = True, update_each_frame: bool = True) -> Dict:
    """Pick the fastest march schedule over `poses` (frames per pose per candidate).
    With `update_each_frame` (the render loop updates the sources every frame) each
    timed frame runs update_buffers first and the score adds its classification time.
    Returns {"choice": {...}, "march_us": {candidate: score in us}}."""
    key = _key(vis)
    if use_cache and key in _CACHE:
        _apply(vis, _CACHE[key])
        return {"choice": dict(_CACHE[key]), "march_us": {}, "cached": True}
    names = ["march_tiles"] + (["march_threads"] if vis.render_form == vis.FORM_COMBINED else [])
    results = {}
    for values in itertools.product(*(CANDIDATES[n] for n in names)):
        _apply(vis, dict(zip(names, values)))
        per_pose = []
        for p in poses:
            vis.look_at = np.asarray(p.look_at, np.float64)
            vis.rotation = np.asarray(p.rotation, np.float64)
            vis.distance = float(p.distance)
            vis._update_modelview()
            vis.draw(out=False)  # warm
            times = []
            for _ in range(frames):
                if update_each_frame:
                    vis.update_buffers()
                vis.draw(out=False)
                t = vis.timings()
                times.append(t["march_us"] + (t["optimization_buffer_us"] if update_each_frame else 0.0))
            per_pose.append(float(np.median(times)))
        # the mean over the poses of each pose's median: every pose weighs the same
        results[values] = (float(np.mean(per_pose)), per_pose)
    best = min(results, key=lambda k: results[k][0])
    choice = dict(zip(names, best))
    _CACHE[key] = choice
    _apply(vis, choice)

    def name(k):
        return ",".join(f"{n[len('march_'):]}={v}" for n, v in zip(names, k))

    return {"choice": dict(choice), "cached": False,
            "march_us": {name(k): t[0] for k, t in results.items()},
            "march_us_per_pose": {name(k): t[1] for k, t in results.items()}}
