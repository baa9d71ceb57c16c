"""The per-source brick arrays of isaac_hip_get_bricks and the layouts behind them (rows of
one source, joint rows of two): what calls between a request, an update and a render may
change, and what they leave alone."""
import numpy as np
import pytest

from isaac_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


def _vis(size=(24, 17, 19), count=2, dtype="F16", fb=(64, 48)):
    """`count` sources (density, vector, soft), all enabled, in the brick form and updated."""
    from isaac_amd import visualization as V

    X, Y, Z = size
    rng = np.random.default_rng(X * 10007 + Y * 101 + Z)
    dens = scenes.gaussian_mixture((Z, Y, X), 5, 6, (0.1 * max(size), 0.3 * max(size))).astype(np.float32)
    vols = [scenes.VolumeSourceSpec("density", dens, "idem", list(scenes.DENSITY_TF), 2.0, 0.4),
            scenes.VolumeSourceSpec("vector", rng.uniform(-0.6, 0.6, (Z, Y, X, 3)).astype(np.float32), "length",
                                    list(scenes.VECTOR_TF), 2.0, 0.0),
            scenes.VolumeSourceSpec("soft", np.ascontiguousarray(1.0 - dens), "idem", list(scenes.DENSITY_TF), 1.5, 0.0)]
    vis = V.from_scene(scenes.SceneSpec("arrays", tuple(size), tuple(size), (1, 1, 1), framebuffer=fb, volumes=vols[:count],
                                        step=0.5, interpolation=True, camera=scenes.FILL_POSE))
    vis.set_render_form(vis.FORM_BRICKS, getattr(vis, dtype))
    vis.update_buffers()
    return vis


def _own(vis):
    """What bricks() gives for both sources of an equal context without joint rows."""
    ref = _vis(vis.local_size, 3)
    out = [ref.bricks(i) for i in (0, 1)]
    ref.close()
    return out


@pytest.mark.parametrize("change", ["smaller", "larger"])
def test_bricks_of_the_last_update_after_a_size_change(change):
    """Asked for between a change of the local size and the next update, joint rows are
    split at the size they were built in."""
    vis = _vis()
    want = _own(vis)
    built = vis.local_size
    vis.update_local_size((9, 8, 7) if change == "smaller" else (64, 64, 64))
    for i in (0, 1):
        pairs, scales = vis.bricks(i)
        assert np.array_equal(pairs, want[i][0]) and np.array_equal(scales, want[i][1])
    vis.update_local_size(built)
    vis.update_buffers()
    for i in (0, 1):
        assert np.array_equal(vis.bricks(i)[0], want[i][0])
    vis.close()


@pytest.mark.parametrize("count", [1, 2])
@pytest.mark.parametrize("built,asked", [("F16", "F32"), ("F32", "F16"), ("F16", "BF16"), ("BF16", "F32")])
def test_brick_type_takes_effect_at_the_next_update(count, built, asked):
    """Frames, batches and bricks() between a change of the brick type and the next update
    read the bricks in the type they were built in."""
    from isaac_amd import batch as B

    vis, other = _vis(count=count, dtype=built), _vis(count=count, dtype=asked)
    want, after = vis.draw(), other.draw()
    arrays = [vis.bricks(i) for i in range(count)]
    b = B.Batch([vis], 64, 48)
    projs, mvs = B.views_for([vis], 1, seed=2)
    ref = vis.draw(projection=projs[0], modelview_=mvs[0])
    vis.set_render_form(vis.FORM_BRICKS, getattr(vis, asked))
    assert np.array_equal(vis.draw(), want)
    for i in range(count):
        for x, y in zip(vis.bricks(i), arrays[i]):
            assert x.dtype == y.dtype and np.array_equal(x, y)
    b.set_views(projs, mvs, bg=vis.background_color)
    b.render(B.GRAPH)
    assert np.array_equal(b.images()[0], ref)
    vis.update_buffers()
    assert np.array_equal(vis.draw(), after)
    b.close()
    vis.close()
    other.close()


@pytest.mark.parametrize("resized", [False, True])
def test_bricks_between_batch_renders(resized):
    """Asking for arrays changes nothing that a batch reads: its next render is accepted and
    gives the same frames, also where the caller's arrays are made anew at another size."""
    from isaac_amd import batch as B

    vis = _vis()
    if resized:
        vis.bricks(0)
        vis.update_local_size((9, 8, 7))
        vis.update_buffers()
    b = B.Batch([vis], 64, 48)
    projs, mvs = B.views_for([vis], 2, seed=2)
    b.set_views(projs, mvs, bg=vis.background_color)
    b.render(B.GRAPH)
    want = b.images()
    for i in (0, 1, 0):
        vis.bricks(i)
        b.render(B.GRAPH)
        assert np.array_equal(b.images(), want), i
    b.close()
    vis.close()


def _pointers(vis, source):
    import ctypes

    from isaac_amd._lib import check, lib

    pairs, scales, n, size = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int64(), ctypes.c_int32()
    check(lib().isaac_hip_get_bricks(vis._ctx, source, ctypes.byref(pairs), ctypes.byref(scales), ctypes.byref(n),
                                     ctypes.byref(size)), vis._ctx, "get_bricks")
    return pairs.value, scales.value


def _enable(vis, slots):
    """The sources' weights and thresholds with all but `slots` switched off."""
    if not hasattr(vis, "all_on"):
        vis.all_on = (list(vis.source_weight), list(vis.iso_threshold))
    vis.source_weight = [w if i in slots else 0.0 for i, w in enumerate(vis.all_on[0])]
    vis.iso_threshold = [t if i in slots else 0.0 for i, t in enumerate(vis.all_on[1])]


def _read(vis, pointers, like):
    vis.synchronize()
    out = [np.empty_like(a) for a in like]
    for a, p in zip(out, pointers):
        vis._d2h(a, p)
    return out


@pytest.mark.parametrize("asked", [(0,), (1,), (0, 1)])
def test_pointers_stay_while_sources_come_and_go(asked):
    """Pointers taken while three sources lie in rows of their own are valid, and hold the
    last update's bricks, when two of them share rows, when one is left and when all are on
    again; nothing is asked for again in between."""
    import torch

    vis = _vis(count=3)
    like = {i: vis.bricks(i) for i in asked}
    held = {i: _pointers(vis, i) for i in asked}
    grow = 1.0
    for slots in ((0, 1), (0,), (0, 1), (1,), (0, 1, 2), (0, 1)):
        _enable(vis, slots)
        grow *= 0.75  # other contents each time
        for s in (0, 1):
            vis.volume_sources[s].tensor.mul_(0.75)
        torch.cuda.synchronize()
        vis.update_buffers()
        vis.draw(out=False)
        for i in asked:
            if i not in slots:
                continue
            pairs, scales = _read(vis, held[i], like[i])
            # a scale is the largest |value| of its brick and component; the pairs are quotients by
            # it, at most 1, which the rounded products move by one step of binary16 at most
            assert np.allclose(scales, like[i][1] * grow, rtol=1e-5), slots
            assert np.abs(pairs.view(np.float16).astype(np.float32) - like[i][0].view(np.float16).astype(np.float32)).max() <= 2.0 ** -11
    for i in asked:
        assert _pointers(vis, i) == held[i]
    vis.close()


def test_switching_a_source_on_and_off_allocates_nothing():
    """Each layout keeps its arrays: once every combination was there, updates neither
    allocate nor free, and the frames are those of the first time."""
    import torch

    vis = _vis(size=(64, 64, 64), count=3)
    cycle = ((0, 1), (0,), (1,), (0, 2), (0, 1, 2))
    frames, free = {}, set()
    for turn in range(3):
        for slots in cycle:
            _enable(vis, slots)
            vis.update_buffers()
            img = vis.draw()
            if turn == 0:
                frames[slots] = img
                continue
            assert np.array_equal(img, frames[slots]), slots
            free.add(torch.cuda.mem_get_info()[0])
    assert len(free) == 1, free
    vis.close()
