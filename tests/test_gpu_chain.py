"""The chain rule's packed step where most Gaussians are hidden and where none
are, at the counts where its workgroups' shares begin and end (64 Gaussians up
to 2^16, then a 1024th of them), and the raw sums cleared only where the pass
before added to them: two steps from different cameras against Oracle B, bit for
bit, parameters, moments and sums."""
import numpy as np
import pytest

from oracle import oracle as O
from vsplat import fixtures as F
import vsplat

pytestmark = pytest.mark.gpu

RATES = vsplat.LearningRates()
RATE_TUPLE = (RATES.position, RATES.scale, RATES.rotation, RATES.opacity, RATES.sh)


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32).reshape(-1)


def _states(t):
    return [t.inspect(f"state_{k}") for k in ("positions", "scales", "rotations", "opacities", "sh")]


def _cloud(count, degree, hidden):
    cloud = F.synthetic_cloud(count, degree, 23, log_scale=(-4.5, 0.4))
    if hidden:  # a wall of opaque splats in front of almost all of the others
        wall = max(1, count // 40)
        cloud.positions[:wall, 2] = -1.5
        cloud.scales[:wall] = np.log(np.float32(0.4))
        cloud.opacities[:wall] = 6.0
        cloud.positions[wall:, 2] = np.abs(cloud.positions[wall:, 2]) * 0.3
        order = np.random.default_rng(count).permutation(count)  # spread over the workgroups
        for name in ("positions", "scales", "rotations", "opacities", "sh"):
            a = getattr(cloud, name)
            a[:] = a.reshape(count, -1)[order].reshape(a.shape)
    return cloud


@pytest.mark.parametrize("hidden", [True, False])
@pytest.mark.parametrize("selective", [True, False])
@pytest.mark.parametrize("count,degree,storage", [(1, 0, vsplat.SH_HALF), (63, 3, vsplat.SH_HALF), (64, 2, vsplat.SH_BF16), (65, 3, vsplat.SH_BF16),
                                                  (129, 1, vsplat.SH_HALF), (4099, 3, vsplat.SH_HALF), (65_536, 1, vsplat.SH_BF16),
                                                  (65_541, 3, vsplat.SH_HALF), (263_000, 0, vsplat.SH_HALF)])
def test_steps_match_the_model(count, degree, storage, selective, hidden):
    cloud = _cloud(count, degree, hidden)
    cams = [F.look_at((0, 0, -3), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 120, 88), F.look_at((0.7, 0.2, -2.8), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 120, 88)]
    target = F.smooth_target(120, 88, 3)
    with vsplat.Trainer(cloud, vsplat.TrainerOptions(force_fixed_point=True, selective_adam=selective, sh_storage=storage)) as t:
        states = [np.zeros_like(s) for s in _states(t)]
        for step, cam in enumerate(cams, 1):
            m = O.Model(t.cloud(), cam, sh_storage=storage)
            r = m.forward()
            m.loss(r, target, 0.2)
            m.backward_fixed(r)
            pos, sc, rot, op, words = m.step(r, RATE_TUPLE, rest_scale=RATES.sh_rest_scale, step=step, selective=selective, states=states)
            t.step(cam, target, RATES)
            np.testing.assert_array_equal(t.inspect("raw"), r.raw_fixed)
            after = t.cloud()
            for got, want in ((after.positions, pos), (after.scales, sc), (after.rotations, rot), (after.opacities, op),
                              (after.sh, F.unpack_sh(words, cloud.coefficients, storage))):
                np.testing.assert_array_equal(_bits(got), _bits(want))
            for got, want in zip(_states(t), states):
                np.testing.assert_array_equal(got, want)
        touched = np.count_nonzero((r.raw_fixed.reshape(count, 14) != 0).any(axis=1))
        print(f"{touched} of {count} touched", flush=True)


@pytest.mark.parametrize("views", [1, 3, 9])
@pytest.mark.parametrize("count,degree,storage", [(1, 0, vsplat.SH_HALF), (65, 3, vsplat.SH_BF16), (1025, 3, vsplat.SH_HALF), (33_000, 1, vsplat.SH_HALF),
                                                  (600_000, 0, vsplat.SH_BF16)])
def test_a_batch_steps_as_its_gradients_applied(count, degree, storage, views):
    """A batch's step, which visits the Gaussians that a view saw, against its summed gradients, stored for all of them, then applied; two in a row."""
    cloud = _cloud(count, degree, True)
    cams = [F.look_at((0.5 * np.sin(k), 0.2 * k, -3 + 0.1 * k), (0, 0, 0), (0.0, -1.0, 0.0), 60.0, 96 + 8 * k, 80) for k in range(views)]
    targets = [F.smooth_target(c.width, c.height, 3 + k) for k, c in enumerate(cams)]
    options = vsplat.TrainerOptions(force_fixed_point=True, sh_storage=storage)
    with vsplat.Trainer(cloud, options) as a, vsplat.Trainer(cloud, options) as b:
        for _ in range(2):
            a.step_views(cams, targets, RATES)
            b.step_views(cams, targets)
            b.apply_gradients(RATES)
            x, y = a.cloud(), b.cloud()
            for name in ("positions", "scales", "rotations", "opacities", "sh"):
                np.testing.assert_array_equal(_bits(getattr(x, name)), _bits(getattr(y, name)))
            for got, want in zip(_states(a), _states(b)):
                np.testing.assert_array_equal(got, want)
            np.testing.assert_array_equal(a.densify_stats(), b.densify_stats())
