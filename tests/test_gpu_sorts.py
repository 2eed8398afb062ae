"""The depth sort and the tile lists at the sizes where the counted passes (one
launch each, tiles of 4096 keys, up to 2^18 keys) and the wide ones past them
begin and end, for depths all different, all equal, mostly out of view and (a near
plane at or behind the camera) negative: the keys sorted, equal keys in
their first order, and each tile's entries in depth order."""
import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


def _check_lists(t, stats):
    keys, values = t.inspect("keys").astype(np.int64), t.inspect("values").astype(np.int64)
    n = len(keys)
    assert np.array_equal(np.sort(values), np.arange(n))
    assert np.array_equal(np.lexsort((values, keys)), np.arange(n))  # sorted by key, equal keys by Gaussian
    assert np.count_nonzero(keys != 0xFFFFFFFF) == stats.visible_splats
    tiles, splats = t.inspect("entry_keys").astype(np.int64), t.inspect("entry_values").astype(np.int64)
    assert len(tiles) == stats.tile_entries
    rank = np.empty(n, np.int64)
    rank[values] = np.arange(n)
    assert np.array_equal(np.lexsort((rank[splats], tiles)), np.arange(len(tiles)))
    ranges = t.inspect("ranges").astype(np.int64)
    assert np.array_equal(ranges[:, 1] - ranges[:, 0], np.bincount(tiles, minlength=len(ranges)))
    assert np.array_equal(np.bincount(splats, minlength=n), _counts(t, rank, stats))


def _counts(t, rank, stats):
    """Each Gaussian's entries, from the offsets in depth order."""
    offsets = t.inspect("coverage").astype(np.int64)
    counts = np.diff(np.append(offsets, stats.tile_entries))
    return counts[rank]


@pytest.mark.parametrize("near", [0.01, 0.0, -5.0])
@pytest.mark.parametrize("scene", ["spread", "equal", "behind"])
@pytest.mark.parametrize("count", [1, 2, 255, 4095, 4096, 4097, 8193, 70_000, 262_143, 262_144, 262_145, 401_409])
def test_depth_order(count, scene, near):
    cloud = F.synthetic_cloud(count, 0, 11, log_scale=(-5.0, 0.5))
    if scene == "equal":
        cloud.positions[:, 2] = 0.25
    if scene == "behind":
        cloud.positions[count // 8:, 2] = -9.0
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 130, 97)
    if scene == "behind" and near <= 0.0:
        cloud.positions[::3, 2] = np.random.default_rng(3).uniform(-7.0, -3.0, len(cloud.positions[::3]))  # negative depths, some kept
        cloud.positions[1::3, 2] = -3.0  # depth 0
        cloud.opacities[:] = -3.0
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(near_plane=near)) as t:
        _check_lists(t, t.compute_gradients(cam, F.smooth_target(130, 97, 3)))


@pytest.mark.parametrize("tiles", [vsplat.TILES_8X8, vsplat.TILES_16X16, vsplat.TILES_32X8, vsplat.TILES_32X32])
@pytest.mark.parametrize("width,height", [(9, 7), (128, 128), (256, 256), (272, 256), (1000, 620), (2500, 1700)])
def test_tile_lists(width, height, tiles):
    """One to three passes over the tile bits, an odd number and an even one, with splats large enough for their own kernels."""
    cloud = F.synthetic_cloud(3000, 0, 13, log_scale=(-4.0, 1.0))
    cloud.scales[::500] = -0.5
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, width, height)
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(tile_shape=tiles)) as t:
        _check_lists(t, t.compute_gradients(cam, F.smooth_target(width, height, 3)))


@pytest.mark.parametrize("tiles", [vsplat.TILES_8X8, vsplat.TILES_16X16, vsplat.TILES_32X8, vsplat.TILES_32X32])
@pytest.mark.parametrize("width,height", [(9, 7), (256, 256), (264, 256), (512, 512), (1000, 620), (1040, 520), (2500, 1700)])
@pytest.mark.parametrize("count,scale", [(3, -2.0), (3000, -4.0), (60_000, -2.5)])
def test_large_tile_lists(count, scale, width, height, tiles):
    """Lists sized for more than 2^18 entries, few or many of which there are, on one to 67k tiles: the one-pass sort's chunks of 8192 and 16384
    entries (up to 2^10 and 2^11 tiles), and the passes of eight bits past them."""
    cloud = F.synthetic_cloud(count, 0, 17, log_scale=(scale, 0.7))
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, width, height)
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(tile_shape=tiles)) as t:
        t.reserve_entries(262_145)
        for _ in range(2):
            _check_lists(t, t.compute_gradients(cam, F.smooth_target(width, height, 3)))
