"""Batch packing of observations against packing world by world: names, order, shapes, types, values."""
import numpy as np
import pytest

from libero_hip import observations as OB, scene as S
from libero_hip.model import Model


def plans():
    spec = OB.ObservableSpec
    yield 'default', OB.default_plan(Model(S.make_scene('c1', 2)))
    yield 'shapes', OB.ObservationPlan((
        spec('scalar', 'a', 'qpos', 1, (0,), shape=()), spec('one', 'a', 'qpos', 1, (1,), shape=(1,)),
        spec('off', 'a', 'qpos', 2, (0, 1), enabled=False, shape=(2,)), spec('three', 'a', 'site_pos', 3, (0,), shape=(3,)),
        spec('pose', 'b', 'inverse_pose', 16, dependencies=('three', 'quat'), shape=(4, 4)),
        spec('hidden', 'b', 'qpos', 2, (2, 3), active=False, shape=(2,))), order=('three', 'scalar', 'one', 'pose'))


@pytest.mark.parametrize('n', [1, 2, 7])
@pytest.mark.parametrize('name', ['default', 'shapes'])
def test_pack_batch_is_the_stack_of_worlds(name, n):
    plan = dict(plans())[name]
    values = np.random.default_rng(n).normal(size=(n, plan.width)).astype(np.float32)
    each = [OB.pack_observations(plan, v) for v in values]
    out = OB.pack_batch(plan, values)
    assert list(out) == list(each[0])
    for k in out:
        want = np.stack([e[k] for e in each])
        assert out[k].dtype == want.dtype and out[k].shape == want.shape and np.array_equal(out[k], want)
        assert not np.shares_memory(out[k], values)
    with pytest.raises(ValueError):
        OB.pack_batch(plan, values[:, 1:])
