"""Downloads at the sizes where they change their way to the host: 96 MiB, past
which they do not go through the pinned slots, and 1 MiB for the statistics."""
import ctypes as C

import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu

UP = (0.0, -1.0, 0.0)


@pytest.mark.parametrize("width,height", [(2500, 2516), (2512, 2512)])
def test_a_large_image(width, height):
    cam = F.look_at((0, 0, -3), (0, 0, 0), UP, 60.0, width, height)
    with vsplat.Trainer(F.synthetic_cloud(500, 1, 3, log_scale=(-2.0, 0.5))) as t:
        for _ in range(2):
            np.testing.assert_array_equal(t.render(cam).view(np.uint32), t.inspect("image").view(np.uint32))


def test_a_large_render_that_does_not_fit_leaves_the_output_alone():
    width, height = 2512, 2512
    cam = F.look_at((0, 0, -3), (0, 0, 0), UP, 60.0, width, height)
    with vsplat.Trainer(F.synthetic_cloud(5000, 0, 3)) as probe:
        needed = probe.gpu_bytes()
    with vsplat.Trainer(F.synthetic_cloud(5000, 0, 3), vsplat.TrainerOptions(memory_budget=needed)) as t:
        out = np.full((width * height, 4), 7.0, np.float32)
        c = vsplat.camera_to_c(cam)
        assert t._lib.vsplat_render(t._h, C.byref(c), vsplat._p(out)) == vsplat.BUDGET_EXCEEDED
        assert (out == 7.0).all()


@pytest.mark.parametrize("count", [32_768, 32_769, 430_000])
def test_gradients_and_statistics(count):
    """The same of each array alone as of all of them together (101 MB at the largest count)."""
    cam = F.look_at((0, 0, -3), (0, 0, 0), UP, 60.0, 97, 63)
    with vsplat.Trainer(F.synthetic_cloud(count, 3, 5), vsplat.TrainerOptions(force_fixed_point=True)) as t:
        t.compute_gradients(cam, F.smooth_target(97, 63, 3))
        np.testing.assert_array_equal(t.densify_stats().view(np.uint32).reshape(-1), t.inspect("stats").view(np.uint32).reshape(-1))
        whole = vars(t.gradients())
        for k, (name, want) in enumerate(whole.items()):
            one = np.full_like(want, np.nan)
            pointers = [None] * 5
            pointers[k] = vsplat._p(one)
            assert t._lib.vsplat_get_gradients(t._h, *pointers) == vsplat.OK
            np.testing.assert_array_equal(one.view(np.uint32), want.view(np.uint32))
        assert np.count_nonzero(whole["positions"]) > 0
