"""The occlusion network's gradient at the edges of its pixel tiles (8 rows x 32
columns per level, 64-pixel rows of the backward-data convolution): one pixel at the
coarsest level, widths and heights around a tile, and batches that leave tiles over."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w", [(1, 8, 8), (3, 8, 40), (2, 72, 24), (1, 64, 256), (5, 32, 264), (2, 136, 64)])
def test_gradient_matches_oracle_per_layer(n, h, w):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from isaac_amd import visualization as V
    from oracle import aonet_oracle as O

    rng = np.random.default_rng(n * 1000 + h + w)
    p = O.init_params(n + h + w)
    f = rng.standard_normal((n, h, w, O.FEATURES)).astype(np.float16).astype(np.float32)
    f[..., 5:] = 0.0
    t = rng.uniform(0.0, 1.0, (n, h, w)).astype(np.float32)
    vis = V.IsaacVisualization("grad", (64, 64), (8, 8, 8), (8, 8, 8), (1, 1, 1), (0, 0, 0), [], [], [])
    vis.aonet_set_params(p)
    loss, g = vis.aonet_loss_grad(f, t)
    again = vis.aonet_loss_grad(f, t)[1]
    vis.close()
    ref_loss, ref = O.loss_and_grad(p.astype(np.float64), f.astype(np.float64), t.astype(np.float64))
    assert abs(loss - ref_loss) <= 2e-3 * ref_loss
    layout, _ = O.param_layout()
    for name, wo, ws, bo, bl in layout:
        # Weights, activations and dz are rounded to binary16 (2^-11 each) in every one of the up to
        # 12 layers in front of and behind a gradient: sqrt(3 * 12 * 2) * 2^-11 / sqrt(3) = 2.4e-3 of
        # it, taken twice.  A unit whose value is within its rounding of 0 can fall on the other
        # side of its ReLU: about one in 1000, which changes one pixel's term in a sum over the P
        # pixels of its level, in one of its channels, 1 / sqrt(P * channels) of that layer's
        # gradient; largest at the coarsest level (64 channels).  (A tap that is missing or
        # doubled at the edge of a tile changes several percent of all terms.)
        tol = 5e-3 + 1.5 / np.sqrt(n * (h // 8) * (w // 8) * 64)
        for part in (slice(wo, wo + int(np.prod(ws))), slice(bo, bo + bl)):
            err = np.linalg.norm(g[part] - ref[part]) / max(np.linalg.norm(ref[part]), 1e-30)
            assert err <= tol, (name, part, err)
        if name != "head":  # the sums of the convolution layers have one order
            assert np.array_equal(g[wo:wo + int(np.prod(ws))], again[wo:wo + int(np.prod(ws))]), name
