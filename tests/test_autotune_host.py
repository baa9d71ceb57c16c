"""The march autotuner's candidate set and choice, on a stub context (no GPU): every
schedule that selects other code is timed once and no other key is touched, the fastest is
kept, and tuning the brick form leaves the combined form's workgroup size alone."""
import numpy as np
import pytest

from isaac_amd import autotune


class _Stub:
    TUNE_MARCH_PREFETCH, TUNE_MARCH_WAVES, TUNE_MARCH_TILES, TUNE_TEX_LAYOUT, TUNE_MARCH_THREADS = 0, 1, 2, 3, 4
    FORM_COMBINED, FORM_BRICKS = 0, 1

    def __init__(self, best, form=0):
        self.render_form = form
        self.framebuffer_size = (64, 32)
        self.local_size = (16, 16, 16)
        self.volume_sources, self.particle_sources = [1], []
        self.interpolation = True
        self.state = {self.TUNE_MARCH_TILES: 4, self.TUNE_MARCH_THREADS: 64}  # the library's defaults
        self.set = set()
        self.tried = []
        self.updates = 0
        self.best = best

    def set_tuning(self, key, value):
        self.set.add(key)
        self.state[key] = value

    def update_buffers(self):
        self.updates += 1

    def _update_modelview(self):
        pass

    def schedule(self):
        return self.state[self.TUNE_MARCH_TILES], self.state[self.TUNE_MARCH_THREADS]

    def draw(self, out=None):
        self.tried.append(self.schedule())

    def timings(self):
        return {"march_us": 100.0 if self.schedule() == self.best else 200.0, "optimization_buffer_us": 10.0}


class _Pose:
    look_at = (0.0, 0.0, 0.0)
    rotation = np.eye(3)
    distance = -4.0


@pytest.mark.parametrize("update_each_frame", [True, False])
def test_schedules_that_differ_are_timed_and_no_other_key_is_set(update_each_frame):
    vis = _Stub(best=(4, 64))
    r = autotune.tune_march(vis, [_Pose()], frames=1, use_cache=False, update_each_frame=update_each_frame)
    assert sorted(set(vis.tried)) == sorted((t, n) for t in (0, 4, 8) for n in (64, 256))
    assert len(vis.tried) == 2 * len(set(vis.tried)) and len(r["march_us"]) == 6
    assert vis.set == {vis.TUNE_MARCH_TILES, vis.TUNE_MARCH_THREADS}
    assert vis.updates == (6 if update_each_frame else 0)


def test_the_fastest_candidate_is_kept():
    vis = _Stub(best=(8, 256))
    r = autotune.tune_march(vis, [_Pose()], frames=2, use_cache=False, update_each_frame=False)
    assert r["choice"] == {"march_tiles": 8, "march_threads": 256}
    assert vis.schedule() == (8, 256)


def test_tuning_the_brick_form_leaves_the_workgroup_size():
    autotune._CACHE.clear()
    vis = _Stub(best=(8, 64), form=_Stub.FORM_BRICKS)
    r = autotune.tune_march(vis, [_Pose()], frames=1, update_each_frame=False)
    assert r["choice"] == {"march_tiles": 8} and vis.set == {vis.TUNE_MARCH_TILES}
    assert {n for _, n in vis.tried} == {64}
    # the cached choice too
    again = autotune.tune_march(vis, [_Pose()], frames=1, update_each_frame=False)
    assert again["cached"] and vis.set == {vis.TUNE_MARCH_TILES} and vis.schedule() == (8, 64)
    autotune._CACHE.clear()
