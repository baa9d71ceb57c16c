"""The brick form's march against its counting variant, which clamps the taps at every
step, at volume sizes about a brick (8 voxels) and its apron, and the batch's work
queues at frame sizes that leave tiles and super-tiles over."""
import dataclasses

import numpy as np
import pytest

from isaac_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


def _spec(size, sources, fb=(141, 99), step=0.5, pose=scenes.FILL_POSE):
    X, Y, Z = size
    rng = np.random.default_rng(X * 10007 + Y * 101 + Z)
    dens = (0.7 * scenes.gaussian_mixture((Z, Y, X), 5, 6, (0.1 * max(size), 0.3 * max(size)))
            + 0.2 * rng.uniform(0.0, 1.0, (Z, Y, X))).astype(np.float32)
    vec = rng.uniform(-0.6, 0.6, (Z, Y, X, 3)).astype(np.float32)
    vols = {"density": scenes.VolumeSourceSpec("density", dens, "idem", list(scenes.DENSITY_TF), 2.0, 0.4),
            "vector": scenes.VolumeSourceSpec("vector", vec, "length", list(scenes.VECTOR_TF), 2.0, 0.0),
            "soft": scenes.VolumeSourceSpec("soft", np.ascontiguousarray(1.0 - dens), "idem", list(scenes.DENSITY_TF), 1.5, 0.0),
            "scaled": scenes.VolumeSourceSpec("scaled", vec, "length | mul(0.8)", list(scenes.VECTOR_TF), 1.0, 0.0)}
    return scenes.SceneSpec("bricks", tuple(size), tuple(size), (1, 1, 1), framebuffer=fb, volumes=[vols[s] for s in sources],
                            step=step, interpolation=True, camera=pose)


@pytest.mark.parametrize("sources", [("density",), ("vector",), ("density", "vector"), ("scaled", "density")])
@pytest.mark.parametrize("size", [(1, 1, 1), (8, 9, 7), (17, 16, 24), (41, 8, 33)])
def test_brick_march_equals_counting_march(size, sources):
    from isaac_amd import visualization as V

    vis = V.from_scene(_spec(size, sources))
    for dtype in (vis.F32, vis.F16, vis.BF16):
        vis.set_render_form(vis.FORM_BRICKS, dtype)
        for step in (0.5, 0.11, 2.5):
            vis.step = step
            vis.update_buffers()
            img = vis.draw()
            g = [a.copy() for a in vis.gbuffer()]
            vis.set_counting(True)
            assert np.array_equal(vis.draw(), img), (dtype, step)
            for a, b in zip(vis.gbuffer(), g):
                assert np.array_equal(a, b), (dtype, step)
            vis.set_counting(False)
    vis.close()


@pytest.mark.parametrize("linear", [True, False])
@pytest.mark.parametrize("dtype", ["F32", "F16", "BF16"])
def test_three_sources_against_the_oracle(oracle_lib, dtype, linear):
    """Three sources (no signature of their own: every one through the general fetch) at a size
    that leaves partial bricks on each axis, within 2/255 of the oracle on 99.9 % of the pixels
    (colours of 8 bits whose sums round in another order)."""
    from isaac_amd import visualization as V
    from oracle import oracle

    spec = dataclasses.replace(_spec((17, 21, 30), ("density", "vector", "soft")), interpolation=linear)
    vis = V.from_scene(spec)
    vis.set_render_form(vis.FORM_BRICKS, getattr(vis, dtype))
    vis.update_buffers()
    img = vis.draw()
    ora = oracle.render_post(spec, 32, getattr(vis, dtype))
    assert (img[..., 3] > 0).mean() > 0.1
    assert (np.abs(img.astype(np.int32) - ora.rgba.astype(np.int32)).max(axis=2) <= 2).mean() >= 0.999
    vis.close()


@pytest.mark.parametrize("fb", [(16, 16), (65, 63), (333, 201), (700, 30)])
def test_batch_frames_of_any_size(fb):
    from isaac_amd import batch as B

    vises, _ = B.make_subvolumes(0, count=3, seed=4, fb=fb, dtype=1, sides=[24, 40, 16])
    projs, mvs = B.views_for(vises, 2, seed=4)
    ref = np.stack([vises[f // 2].draw(projection=projs[f], modelview_=mvs[f]) for f in range(6)])
    b = B.Batch(vises, *fb)
    b.set_views(projs, mvs, bg=vises[0].background_color)
    for chunk, groups in ((1, 4), (3, 1), (64, 2)):
        b.set_tuning(B.TUNE_CHUNK, chunk)
        b.set_tuning(B.TUNE_GROUPS_PER_CU, groups)
        b.render(B.GRAPH)
        assert np.array_equal(b.images(), ref), (chunk, groups)
    b.close()
    for v in vises:
        v.close()


@pytest.mark.parametrize("dtype", ["F16", "BF16"])
@pytest.mark.parametrize("sources", [("density", "vector"), ("scaled", "density"), ("density", "soft")])
@pytest.mark.parametrize("size", [(1, 1, 1), (8, 9, 7), (17, 16, 24), (41, 8, 33)])
def test_joint_rows_equal_rows_of_one_source(size, sources, dtype):
    """Two sources in joint rows against the same two in rows of their own (update_buffers
    with a third source enabled keeps every source apart; it is switched off after it), one
    of two joined sources against the same in its own rows, and the arrays that bricks()
    gives for a joined source before and after another update against those of its own."""
    from isaac_amd import visualization as V

    spec = _spec(size, sources + ("vector",))
    spec.volumes[2] = dataclasses.replace(spec.volumes[2], name="third")
    vis = V.from_scene(spec)
    vis.set_render_form(vis.FORM_BRICKS, getattr(vis, dtype))
    weights, iso = list(vis.source_weight), list(vis.iso_threshold)

    def enable(slots):
        vis.source_weight = [w if i in slots else 0.0 for i, w in enumerate(weights)]
        vis.iso_threshold = [t if i in slots else 0.0 for i, t in enumerate(iso)]

    def frame():
        img = vis.draw()
        return [img] + [a.copy() for a in vis.gbuffer()]

    def same(a, b):
        return all(np.array_equal(x, y) for x, y in zip(a, b))

    enable((0, 1, 2))
    vis.update_buffers()
    own = [vis.bricks(i) for i in (0, 1)]
    want = {}
    for slots in ((0, 1), (0,), (1,)):
        enable(slots)
        want[slots] = frame()
    enable((0, 1))
    vis.update_buffers()
    for slots in want:
        enable(slots)
        assert same(frame(), want[slots]), slots
    enable((0, 1))
    for again in range(3):
        for i in (0, 1):
            pairs, scales = vis.bricks(i)
            assert np.array_equal(pairs, own[i][0]) and np.array_equal(scales, own[i][1]), (again, i)
        vis.update_buffers()
        assert same(frame(), want[(0, 1)])
    vis.close()
