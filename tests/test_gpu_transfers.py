"""Downloads through pinned slots, at the sizes where their chunks (1 MiB), slots
(12) and helper threads (from 3 MiB) begin and end; uploads beside the passes;
and the status a pass leaves for the calls that read it."""
import ctypes as C

import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(16, 16), (256, 255), (256, 256), (257, 256), (512, 383), (512, 384), (1024, 767), (1024, 768),
                                          (1024, 833), (1037, 1631)])
def test_render_downloads_the_image(width, height):
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, width, height)
    with vsplat.Trainer(F.synthetic_cloud(500, 1, 3, log_scale=(-2.0, 0.5))) as t:
        for _ in range(2):
            np.testing.assert_array_equal(t.render(cam).view(np.uint32), t.inspect("image").view(np.uint32))


@pytest.mark.parametrize("count,degree", [(1, 0), (700, 3), (4444, 3), (17_000, 3), (71_003, 2)])
def test_cloud_and_gradients_come_back_whole(count, degree):
    """The parameters as uploaded (their SH representable as halves), and gradients that agree between two ways of asking."""
    cloud = F.synthetic_cloud(count, degree, 5, sh_sigma=0.3 if degree else None)
    cloud.sh[:] = cloud.sh.astype(np.float16).astype(np.float32)
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 97, 63)
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True)) as t:
        back = t.cloud()
        for name in ("positions", "scales", "rotations", "opacities", "sh"):
            np.testing.assert_array_equal(getattr(back, name), getattr(cloud, name))
        t.compute_gradients(cam, F.smooth_target(97, 63, 3))
        g = t.gradients()
        for k, name in enumerate(("positions", "scales", "rotations", "opacities", "sh")):
            one = np.zeros_like(getattr(g, name))
            args = [None] * 5
            args[k] = vsplat._p(one)
            assert t._lib.vsplat_get_gradients(t._h, *args) == vsplat.OK
            np.testing.assert_array_equal(one.view(np.uint32), getattr(g, name).view(np.uint32))
        assert np.count_nonzero(g.positions) > 0


def test_a_render_that_does_not_fit_leaves_the_output_alone():
    cam = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 640, 480)
    with vsplat.Trainer(F.synthetic_cloud(5000, 0, 3)) as probe:
        needed = probe.gpu_bytes()
    with vsplat.Trainer(F.synthetic_cloud(5000, 0, 3), vsplat.TrainerOptions(memory_budget=needed)) as t:
        out = np.full((640 * 480, 4), 7.0, np.float32)
        c = vsplat.camera_to_c(cam)
        assert t._lib.vsplat_render(t._h, C.byref(c), vsplat._p(out)) == vsplat.BUDGET_EXCEEDED
        assert (out == 7.0).all()


def test_status_of_queued_steps():
    """A queued step that does not fit is reported once; a render into GPU memory in between does not take its place."""
    cloud, cam = F.synthetic_cloud(5000, 0, 3), F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 320, 240)
    small = F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 16, 16)
    target, out = vsplat.DeviceBuffer(F.smooth_target(320, 240, 3)), vsplat.DeviceBuffer.empty(320 * 240 * 16)
    with vsplat.Trainer(cloud) as t:
        t.reserve_entries(16)
        t.enqueue(cam, target.ptr, vsplat.MODE_GRADIENTS)
        t.render_noalloc(small, out)
        with pytest.raises(RuntimeError):
            t.synchronize()
        t.synchronize()
        want = t.compute_gradients(cam, F.smooth_target(320, 240, 3))
        t.enqueue(cam, target.ptr, vsplat.MODE_GRADIENTS)
        t.render_noalloc(small, out)
        got = t.synchronize()
        assert (got.loss, got.visible_splats, got.tile_entries) == (want.loss, want.visible_splats, want.tile_entries)
