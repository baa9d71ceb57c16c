"""The combined form's march against its counting variant, which tests the iso alpha
and clamps the texels at every step: volumes about the sizes of a texel, of an iso
cell (8 texels) and of several, where the interior steps and the marked cells begin
and end, and the states an iso texture can be in between updates."""
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


def _spec(size, linear=True, iso=0.4, step=0.5, pose=scenes.DEFAULT_POSE):
    X, Y, Z = size
    rng = np.random.default_rng(X * 10007 + Y * 101 + Z)
    dens = (0.7 * scenes.gaussian_mixture((Z, Y, X), 5, 6, (0.08 * max(size), 0.3 * max(size)))
            + 0.2 * rng.uniform(0.0, 1.0, (Z, Y, X))).astype(np.float32)
    vol = scenes.VolumeSourceSpec("density", dens, "idem", list(scenes.DENSITY_TF), 2.0, iso)
    return scenes.SceneSpec("march", tuple(size), tuple(size), (1, 1, 1), framebuffer=(150, 117), volumes=[vol], step=step,
                            interpolation=linear, camera=pose, clipping=[((0.1, 0.0, 0.0), (1.0, 0.2, 0.0))])


def _counting_equal(vis):
    img = vis.draw()
    g = [a.copy() for a in vis.gbuffer()]
    vis.set_counting(True)
    ref = vis.draw()
    gr = [a.copy() for a in vis.gbuffer()]
    vis.set_counting(False)
    assert np.array_equal(img, ref)
    for a, b in zip(g, gr):
        assert np.array_equal(a, b)
    return img


@pytest.mark.parametrize("linear", [True, False])
@pytest.mark.parametrize("size", [(1, 1, 1), (2, 1, 3), (7, 8, 9), (16, 17, 15), (40, 8, 23), (8, 64, 8), (65, 33, 49)])
def test_march_equals_counting_march(size, linear):
    from isaac_amd import visualization as V

    for step, pose in ((0.5, scenes.FILL_POSE), (0.13, scenes.Camera(distance=-1.2)), (3.0, scenes.DEFAULT_POSE)):
        vis = V.from_scene(_spec(size, linear, step=step, pose=pose))
        for iso in (0.4, 0.05, 0.0):
            vis.iso_threshold = [iso]
            vis.update_buffers()
            _counting_equal(vis)
        vis.close()


@pytest.mark.parametrize("linear", [True, False])
@pytest.mark.parametrize("data", ["full", "noise", "dots", "slabs"])
def test_rays_that_start_in_marked_cells(data, linear):
    """Data with a surface everywhere: all above the threshold, noise about it, single voxels
    above it 5 apart (marked throughout, hardly a hit), and slabs of 24 voxels above and below
    it (rays start in fewer marked cells in a row), along a box of 16 iso cells and more."""
    from isaac_amd import visualization as V

    X, Y, Z = 150, 52, 141
    z, y, x = np.meshgrid(np.arange(Z), np.arange(Y), np.arange(X), indexing="ij")
    dens = {"full": np.full((Z, Y, X), 0.9), "noise": np.random.default_rng(3).uniform(0.0, 1.0, (Z, Y, X)),
            "dots": np.where((x % 5 == 2) & (y % 5 == 2) & (z % 5 == 2), 0.55, 0.0),
            "slabs": np.where((x + y) // 24 % 2 == 0, 0.8, 0.1)}[data].astype(np.float32)
    spec = _spec((X, Y, Z), linear, pose=scenes.FILL_POSE)
    spec.volumes[0] = dataclasses.replace(spec.volumes[0], data=dens)
    vis = V.from_scene(spec)
    hits = 0
    for step in (0.5, 2.5):
        vis.step = step
        for iso in (0.5, 0.05):
            vis.iso_threshold = [iso]
            vis.update_buffers()
            _counting_equal(vis)
            hits += int((vis.gbuffer()[1] < 3e38).sum())
    assert hits > (0 if data == "dots" else 1000)  # (a trilinear sum about a single voxel hardly reaches the threshold)
    vis.close()


def test_iso_threshold_changed_between_updates():
    """A threshold set after a classification without one finds no surface until the next
    update, as the iso texels are 0 then; the texels a caller asked for follow every update."""
    from isaac_amd import visualization as V

    vis = V.from_scene(_spec((24, 20, 16), iso=0.0))
    vis.update_buffers()
    plain = _counting_equal(vis)
    vol, iso = vis.combined_textures()
    assert not iso.any() and vol.any()
    vis.iso_threshold = [0.3]
    assert np.array_equal(_counting_equal(vis), plain)
    vis.update_buffers()
    assert not np.array_equal(_counting_equal(vis), plain)
    vol2, iso2 = vis.combined_textures()
    assert iso2.any() and np.array_equal(vol, vol2)
    vis.iso_threshold = [0.0]
    vis.update_buffers()
    assert np.array_equal(_counting_equal(vis), plain)
    assert not vis.combined_textures()[1].any()
    vis.close()


def test_surfaces_around_the_wrap_of_the_marks():
    """The marks of the iso cells carry their update's number, 1..255 in turn, and are cleared
    when it wraps: the surface of every update about two wraps, another one each time, is
    the counting march's, which does not read the marks.  (A mark that outlived its update would
    only have steps tested in vain; a lost one would lose the surface.)"""
    from isaac_amd import visualization as V

    vis = V.from_scene(dataclasses.replace(_spec((24, 20, 16)), clipping=[]))
    plain, frames = None, []
    for k in range(1, 516):  # update k has number (k - 1) % 255 + 1
        near = min(k % 255, 255 - k % 255) <= 4
        vis.iso_threshold = [(0.4, 0.2, 0.6)[k % 3] if near else 0.0]
        vis.update_buffers()
        if near:
            frames.append(_counting_equal(vis))
        elif plain is None:
            plain = vis.draw()
    assert len(frames) > 20 and all(not np.array_equal(f, plain) for f in frames)
    assert np.array_equal(frames[-1], frames[-4]) and not np.array_equal(frames[-1], frames[-2])
    vis.close()


def test_local_size_that_does_not_fit():
    """A local size whose textures cannot be allocated: an error, then nothing to draw, classify
    or ask for, until a size that fits."""
    import ctypes

    from isaac_amd import visualization as V
    from isaac_amd._lib import IsaacHipError, lib

    vis = V.from_scene(_spec((24, 20, 16)))
    vis.update_buffers()
    want = vis.draw()
    vis.combined_textures()
    with pytest.raises(IsaacHipError):
        vis.update_local_size((1 << 20, 1 << 13, 1 << 12))  # 2^45 voxels: 256 TiB
    for call in (vis.draw, vis.update_buffers):
        with pytest.raises(IsaacHipError):
            call()
    ptr, size = ctypes.c_void_p(1), ctypes.c_int32()
    assert lib().isaac_hip_get_combined_textures(vis._ctx, ctypes.byref(ptr), ctypes.byref(size)) == 0
    assert not ptr.value and size.value == 8
    vis.update_local_size((24, 20, 16))
    vis.update_buffers()
    assert np.array_equal(vis.draw(), want)
    vol, iso = vis.combined_textures()
    assert vol.any() and iso.any()
    vis.close()
