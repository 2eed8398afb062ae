"""vsplat_render_noalloc at the numbers of tiles where the tile sort, and with it
the scratch it takes, changes: one layout serves them all."""
import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(256, 256), (264, 256), (512, 256), (512, 264), (2048, 1024)])
def test_renders_on_either_side_of_a_tile_sort(width, height):
    """1024, 1056, 2048, 2112 and 32768 tiles of 8x8, in turn in one trainer and on the same scratch."""
    cloud = F.synthetic_cloud(20_000, 1, 3, log_scale=(-4.0, 0.5))
    cam, other = (F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, w, h) for w, h in ((width, height), (640, 480)))
    out = vsplat.DeviceBuffer(np.full(width * height * 4 + 640 * 480 * 4, np.nan, np.float32))
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(tile_shape=vsplat.TILES_8X8)) as t:
        for c in (cam, other, cam):
            t.render_noalloc(c, out)
            got = out.read(np.float32)[: c.width * c.height * 4]
            np.testing.assert_array_equal(got.view(np.uint32), t.render(c).reshape(-1).view(np.uint32))
    out.free()
