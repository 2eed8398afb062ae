"""Batches of views: what a refused one leaves behind, batches beside single
steps, and the batched chain rule where few, about half and all of the Gaussians
are seen, with the options that act on the ones no view saw."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
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


NAMES = ("positions", "scales", "rotations", "opacities", "sh")
RATE_TUPLE = (RATES.position, RATES.scale, RATES.rotation, RATES.opacity, RATES.sh)


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32).reshape(-1)


def _states(t):
    return [t.inspect(f"state_{k}") for k in NAMES]


@pytest.mark.parametrize("options", [{}, {"selective_adam": False}, {"opacity_reg": 0.5, "scale_reg": 0.25}, {"active": 1},
                                     {"selective_adam": False, "opacity_reg": 0.5, "active": 2}],
                         ids=["plain", "every parameter", "penalties", "degree 1", "all of them"])
@pytest.mark.parametrize("views,storage", [(2, vsplat.SH_HALF), (9, vsplat.SH_BF16)])
@pytest.mark.parametrize("seen", [0.04, 0.5, 0.62, 1.0])
def test_batches_by_the_share_seen(seen, views, storage, options):
    """Gradients and a step of a batch against Oracle B's summed gradients and its Adam, and a second step against the gradients stored, then applied.
    Workgroups of 64 Gaussians, whose shares seen lie on both sides of where a whole workgroup is listed."""
    count, degree = 1217, 3
    active = options.get("active", degree)
    given = {k: v for k, v in options.items() if k != "active"}
    regs = {k: given.get(k, 0.0) for k in ("opacity_reg", "scale_reg")}
    selective = given.get("selective_adam", True)
    rng = np.random.default_rng(7)
    cloud = F.synthetic_cloud(count, degree, 23, log_scale=(-3.5, 0.4), sh_sigma=0.3)
    cloud.positions[:] = rng.uniform(-0.6, 0.6, (count, 3)).astype(np.float32)
    cloud.positions[rng.permutation(count)[round(seen * count):], 2] = -9.0  # behind every camera
    cloud.opacities[:] = -2.0
    cams = _cameras([(72 + 8 * (k % 3), 56) for k in range(views)])
    targets = [F.smooth_target(c.width, c.height, 3 + k) for k, c in enumerate(cams)]
    total, stats = None, np.zeros((count, 8), np.float32)
    for cam, target in zip(cams, targets):
        m = O.Model(cloud, cam, active_degree=active, sh_storage=storage)
        r = m.forward()
        m.loss(r, target, 0.2)
        m.backward_fixed(r)
        g, stats = m.gradients(r, stats=stats, **regs)
        total = [x.copy() for x in g] if total is None else [a + b for a, b in zip(total, g)]
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, sh_storage=storage, **given)) as a, \
         vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, sh_storage=storage, **given)) as b:
        for t in (a, b):
            t.set_active_sh_degree(active)
        uploaded = a.cloud()
        states = [np.zeros_like(s) for s in _states(a)]
        pos, sc, rot, op, words = O.adam_from_gradients(uploaded, m.words, total, RATE_TUPLE, rest_scale=RATES.sh_rest_scale, selective=selective,
                                                        sh_storage=storage, states=states)
        b.step_views(cams, targets)
        for name, want in zip(NAMES, total):
            np.testing.assert_array_equal(_bits(getattr(b.gradients(), name)), _bits(want))
        np.testing.assert_array_equal(_bits(b.densify_stats()), _bits(stats))
        b.apply_gradients(RATES)
        a.step_views(cams, targets, RATES)
        after = a.cloud()
        for name, want in zip(NAMES, (pos, sc, rot, op, F.unpack_sh(words, cloud.coefficients, storage))):
            np.testing.assert_array_equal(_bits(getattr(after, name)), _bits(want))
        for got, want in zip(_states(a), states):
            np.testing.assert_array_equal(got, want)
        a.step_views(cams, targets, RATES)
        b.step_views(cams, targets)
        b.apply_gradients(RATES)
        for name in NAMES:
            np.testing.assert_array_equal(_bits(getattr(a.cloud(), name)), _bits(getattr(b.cloud(), name)))
        for got, want in zip(_states(a), _states(b)):
            np.testing.assert_array_equal(got, want)


def test_a_step_over_views_leaves_the_stored_gradients():
    cloud, cams = F.synthetic_cloud(3000, 2, 3, log_scale=(-2.0, 0.5)), _cameras([(72, 56), (96, 40)])
    targets = [F.smooth_target(c.width, c.height, 3 + k) for k, c in enumerate(cams)]
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True)) as t:
        t.compute_gradients(cams[0], targets[0])
        before = vars(t.gradients())
        t.step_views(cams, targets, RATES)
        for name, got in vars(t.gradients()).items():
            np.testing.assert_array_equal(_bits(got), _bits(before[name]))


@pytest.mark.parametrize("sizes", [[(352, 360), (360, 368)], [(360, 368), (440, 440), (448, 448)]])
def test_batches_on_either_side_of_the_launch_rule(sizes):
    """Views of 1984 to 3136 8x8 blocks: four waves a block up to 2048 in a batch and up to 3072 alone; image and sums are those of the view alone."""
    cloud, cams = F.random_cloud(600, 1, 11), [F.train_camera(w, h) for w, h in sizes]
    targets = [F.smooth_target(c.width, c.height, 3) for c in cams]
    options = vsplat.TrainerOptions(force_fixed_point=True, tile_shape=vsplat.TILES_8X8)
    with vsplat.Trainer(cloud, options) as t, vsplat.Trainer(cloud, options) as one:
        t.step_views(cams, targets)
        for k, (cam, target) in enumerate(zip(cams, targets)):
            one.compute_gradients(cam, target)
            np.testing.assert_array_equal(_bits(t.inspect("image", view=k)), _bits(one.inspect("image")))
            np.testing.assert_array_equal(t.inspect("raw", view=k), one.inspect("raw"))
            assert np.count_nonzero(one.inspect("raw")) > 0


@pytest.mark.parametrize("views", [2, 8, 9])
def test_memory_of_a_trainer_that_steps_batches(views):
    """A step holds the SH sums, or for more views than the chain rule takes at once the gradients, and not both."""
    cloud, cams = F.synthetic_cloud(30_000, 3, 3), _cameras([(48, 40)] * views)
    targets = [F.smooth_target(48, 40, 3)] * views
    held = []
    for rates in (None, RATES):
        with vsplat.Trainer(cloud) as t:
            t.step_views(cams, targets, rates)
            held.append(t.gpu_bytes())
    assert held[0] - held[1] == (30_000 * 4 * 11 if views <= 8 else 0)
