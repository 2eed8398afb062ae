"""The raster passes' walk over a tile's list, at the lengths where its batches
of 64 or 256 entries and its groups and chunks of splats end, and its staging of
long, thin splats that cross the 8x8 blocks at an angle: images and fixed-point
sums bit for bit against Oracle B, whose lists are 16x16 and which stages
nothing. On views of few blocks, each worked by four waves, and of more than
3072, each worked by one."""
import numpy as np
import pytest

from oracle import oracle as O
from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _check(cloud, cam, target, **options):
    model = O.Model(cloud, cam)
    r = model.forward()
    model.loss(r, target, 0.2)
    model.backward_fixed(r)
    t = vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, **options))
    t.compute_gradients(cam, target)
    np.testing.assert_array_equal(_bits(t.inspect("image")), _bits(r.image))
    np.testing.assert_array_equal(t.inspect("raw"), r.raw_fixed)
    return r


@pytest.mark.parametrize("tiles", [vsplat.TILES_16X16, vsplat.TILES_8X8, vsplat.TILES_32X32])
@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("logit", [-3.0, 2.0])
@pytest.mark.parametrize("count", [1, 3, 4, 5, 63, 64, 65, 68, 128, 129, 257])
def test_list_lengths(count, logit, recompute, tiles):
    """`count` splats over the same pixels: nearly transparent, so that every pixel walks the whole list, or opaque enough to stop."""
    cloud = F.random_cloud(count, 1, 5)
    rng = np.random.default_rng(count)
    cloud.positions[:] = rng.uniform(-0.15, 0.15, (count, 3)).astype(np.float32) + np.array([0, 0, 4], np.float32)
    cloud.opacities[:] = logit
    cloud.scales[:] = np.log(rng.uniform(0.05, 0.3, (count, 3))).astype(np.float32)
    r = _check(cloud, F.train_camera(43, 37), F.smooth_target(43, 37, 3), recompute_transmittance=recompute, tile_shape=tiles)
    assert (r.ranges[:, 1] - r.ranges[:, 0]).max() == count


@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("logit", [-3.0, 2.0])
@pytest.mark.parametrize("count", [1, 4, 5, 64, 65, 129, 257])
def test_list_lengths_with_a_wave_a_block(count, logit, recompute):
    """As above on a view of 3136 blocks; the splats cover the 8x8 blocks at the middle of the view."""
    cloud = F.random_cloud(count, 1, 5)
    rng = np.random.default_rng(count)
    cloud.positions[:] = rng.uniform(-0.01, 0.01, (count, 3)).astype(np.float32) + np.array([0, 0, 4], np.float32)
    cloud.opacities[:] = logit
    cloud.scales[:] = np.log(rng.uniform(0.01, 0.06, (count, 3))).astype(np.float32)
    r = _check(cloud, F.train_camera(448, 448), F.smooth_target(448, 448, 3), recompute_transmittance=recompute)
    assert (r.ranges[:, 1] - r.ranges[:, 0]).max() == count


@pytest.mark.parametrize("tiles", [vsplat.TILES_16X16, vsplat.TILES_8X8, vsplat.TILES_32X8, vsplat.TILES_32X32])
@pytest.mark.parametrize("width,height", [(8, 8), (1, 1), (280, 280), (288, 288), (376, 512), (384, 512), (392, 512)])
def test_views_at_the_edges_of_the_launch_rules(width, height, tiles):
    """One block, around 1280 (ordered backward) and around 3072 blocks (a wave a block), in each tile shape; sums with and without the two scores."""
    cloud = F.random_cloud(600, 1, 11)
    cam, target = F.train_camera(width, height), F.smooth_target(width, height, 3)
    _check(cloud, cam, target, tile_shape=tiles)
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, tile_shape=tiles)) as t:
        stats = t.score_view(cam, target, 0.5, 2.0)
        got = t.densify_stats()
    m = O.Model(cloud, cam)
    r = m.forward()
    m.loss(r, target, 0.2, score_share=0.5)
    m.backward_fixed(r)
    np.testing.assert_array_equal(_bits(got), _bits(O.score_statistics(m.statistics(r), r.raw, 3.0 * width * height * 2.0, stats.loss)))


@pytest.mark.parametrize("tiles", [vsplat.TILES_16X16, vsplat.TILES_32X8, vsplat.TILES_32X32])
@pytest.mark.parametrize("length,thin", [(1.0, 0.003), (20.0, 0.03), (200.0, 0.05), (600.0, 0.3)])
def test_long_thin_splats(length, thin, tiles):
    """Splats whose conic's terms cancel, at many angles: staging must keep each in every block one of whose pixels takes it."""
    count = 48
    cloud = F.random_cloud(count, 1, 7)
    angle = np.linspace(0.0, np.pi, count) / 2
    cloud.rotations[:] = np.stack([np.cos(angle), 0 * angle, 0 * angle, np.sin(angle)], 1)
    cloud.scales[:] = np.log(np.array([length, thin, thin], np.float32))
    cloud.opacities[:] = 0.5
    _check(cloud, F.train_camera(150, 118), F.smooth_target(150, 118, 3), tile_shape=tiles)
