"""Splats so large that their 2D determinant overflows: their conic is zero, and
every tile shape draws them in the same pixels."""
import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(120, 88), (520, 440)])
@pytest.mark.parametrize("recompute", [False, True])
def test_a_zero_conic_in_every_tile_shape(recompute, width, height):
    """On a view of few blocks, worked by four waves each, and on one of 3575."""
    cloud = F.random_cloud(60, 1, 13)
    large = np.arange(3, 60, 7)
    for i, log_scale in zip(large, (21.0, 22.0, 23.0, 24.0, 30.0, 41.0, 42.0, 42.8, 43.3)):
        cloud.positions[i] = [0.3 * (i - 30) / 30, 0.05, 3.5 + 0.01 * i]
        cloud.scales[i] = log_scale
        cloud.opacities[i] = -1.0
    cam, target = F.train_camera(width, height), F.smooth_target(width, height, 3)
    images, sums = [], []
    for tiles in (vsplat.TILES_8X8, vsplat.TILES_16X16, vsplat.TILES_32X8, vsplat.TILES_32X32):
        with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, recompute_transmittance=recompute, tile_shape=tiles)) as t:
            t.compute_gradients(cam, target)
            conics = t.inspect("splats").view(np.float32).reshape(-1, 12)[:, :3]
            images.append(t.inspect("image").view(np.uint32))
            sums.append(t.inspect("raw"))
        assert (conics[large] == 0).all(axis=1).sum() >= 2
    for image, raw in zip(images[1:], sums[1:]):
        np.testing.assert_array_equal(image, images[0])
        np.testing.assert_array_equal(raw, sums[0])
    assert np.count_nonzero(sums[0].reshape(60, 14)[large]) > 0
