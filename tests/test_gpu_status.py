"""What a trainer says of itself: the status a queued pass leaves in host memory,
where its cloud is replaced before anybody has asked for it, and the memory it
holds."""
import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fits", [True, False])
def test_a_changed_cloud_has_no_status(fits):
    cloud, cam = F.synthetic_cloud(5000, 0, 3), F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 320, 240)
    target = vsplat.DeviceBuffer(F.smooth_target(320, 240, 3))
    with vsplat.Trainer(cloud) as t:
        t.reserve_entries(1 << 20 if fits else 16)
        t.enqueue(cam, target.ptr, vsplat.MODE_GRADIENTS)
        t.apply_changes(None, np.arange(4000, dtype=np.int64))
        stats = t.synchronize()
        assert (stats.visible_splats, stats.tile_entries) == (0, 0)
        assert t.compute_gradients(cam, F.smooth_target(320, 240, 3)).visible_splats > 0


@pytest.mark.parametrize("count", [1, 5000])
def test_the_sorts_digit_counts_are_memory_too(count):
    """Per tile of 4096 keys and pass 256 words: four passes over the Gaussians, three over at most 2^18 tile entries."""
    words = 4 * -(-count // 4096) * 256 + 3 * 64 * 256
    with vsplat.Trainer(F.synthetic_cloud(count, 0, 3)) as t:
        assert t.gpu_bytes() - t.bytes_per_gaussian() * count >= 4 * words
