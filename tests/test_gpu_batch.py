"""Batches of views: what a refused one leaves behind."""
import ctypes as C

import numpy as np
import pytest

from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu

RATES = vsplat.LearningRates()
UP = (0.0, -1.0, 0.0)


def _cameras(sizes):
    return [F.look_at((0.5 * np.sin(k), 0.2 * k, -3 + 0.1 * k), (0, 0, 0), UP, 60.0, w, h) for k, (w, h) in enumerate(sizes)]


def _step_views(t, cams, targets, sizes):
    n = len(cams)
    c = (vsplat.CCamera * n)(*[vsplat.camera_to_c(x) for x in cams])
    pointers = (C.c_void_p * n)(*[a.ctypes.data for a in targets])
    return t._lib.vsplat_step_views(t._h, n, c, pointers, (C.c_size_t * n)(*sizes), vsplat.MODE_GRADIENTS, None, None)


@pytest.mark.parametrize("wrong", [lambda size, first: size - 4, lambda size, first: 0, lambda size, first: 2**64 - 1,
                                   lambda size, first: 2**64 - first, lambda size, first: 2**63], ids=["less", "none", "most", "wraps", "huge"])
@pytest.mark.parametrize("at", [0, 1])
def test_a_target_of_the_wrong_size_is_refused(at, wrong):
    """Wherever it stands and however the sizes add up, the call says that the target does not match; the next batch is as if it had not been made."""
    cloud, cams = F.synthetic_cloud(3000, 1, 3, log_scale=(-2.0, 0.5)), _cameras([(72, 56), (96, 40)])
    targets = [F.smooth_target(c.width, c.height, 3 + k) for k, c in enumerate(cams)]
    sizes = [t.nbytes for t in targets]
    options = vsplat.TrainerOptions(force_fixed_point=True)
    with vsplat.Trainer(cloud, options) as a, vsplat.Trainer(cloud, options) as b:
        bad = list(sizes)
        bad[at] = wrong(sizes[at], sizes[1 - at])
        assert _step_views(b, cams, targets, bad) == vsplat.RUNTIME_ERROR
        assert b"does not match" in b._lib.vsplat_last_error()
        assert _step_views(a, cams, targets, sizes) == vsplat.OK and _step_views(b, cams, targets, sizes) == vsplat.OK
        for got, want in zip(vars(b.gradients()).values(), vars(a.gradients()).values()):
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
        assert np.count_nonzero(b.gradients().positions) > 0


def test_batches_of_more_views_after_single_steps():
    """The stream that uploads targets makes room for the views' streams and comes back: single calls and batches in turn, each against a trainer of its own."""
    cloud = F.synthetic_cloud(3000, 1, 3, log_scale=(-2.0, 0.5))
    options = vsplat.TrainerOptions(force_fixed_point=True)
    with vsplat.Trainer(cloud, options) as t:
        for views in (0, 2, 0, 4, 3, 0):
            cams = _cameras([(72 + 8 * k, 56) for k in range(max(views, 1))])
            targets = [F.smooth_target(c.width, c.height, 3 + k + views) for k, c in enumerate(cams)]
            with vsplat.Trainer(cloud, options) as fresh:
                for x in (t, fresh):
                    if views == 0:
                        x.compute_gradients(cams[0], targets[0])
                    else:
                        x.step_views(cams, targets)
                for got, want in zip(vars(t.gradients()).values(), vars(fresh.gradients()).values()):
                    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
