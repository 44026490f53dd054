"""The LDS route's two-wave kernel: the same worlds bit for bit at any place and size of a batch, on
both precisions, and to FP32 rounding the workspace route's result (one substep: positions 1e-6,
velocities and accelerations by their scale 1e-4, the parity bar of the two routes)."""
import numpy as np
import pytest

from helpers import rel_err
from test_gpu_wide_kernel import FIELDS
from libero_hip import native, scene as S
from libero_hip.model import Model

pytestmark = pytest.mark.gpu


def run(name, nworld, flags, substeps):
    import torch
    sc = S.make_scene(name, 8, seed=4)
    for k in range((sc.init_qpos.shape[1] - 9) // 7):
        sc.init_qpos[:, 11 + 7 * k] -= 0.0051
    pick = np.arange(nworld) % 8
    m = Model(sc)
    d = native.DeviceData(native.DeviceModel(m), nworld)
    rng = np.random.default_rng(5)
    d['qpos'].copy_(torch.from_numpy(sc.init_qpos[pick]))
    d['osc_gains'].copy_(torch.from_numpy(np.tile(np.r_[sc.osc['kp'], sc.osc['kd']], (nworld, 1))))
    d['osc_q0'].copy_(torch.from_numpy(np.tile(np.asarray(sc.osc['q0'], float), (nworld, 1))))
    d['osc_action'].copy_(torch.from_numpy(rng.uniform(-1, 1, (8, 7))[pick]))
    d['body_active'].fill_(1)
    d.forward(None, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL | flags)
    d.control_step(substeps, native.FLAG_POLICY_FIRST | flags)
    torch.cuda.synchronize()
    return {k: d[k].cpu().numpy() for k in FIELDS}


@pytest.mark.parametrize('route', ['lds', 'fp64'])
@pytest.mark.parametrize('name', ['c1', 'c3'])
def test_two_waves(gpu_available, name, route):
    flags = native.FLAG_LDS if route == 'lds' else native.FLAG_FP64
    print('case', name, route, flush=True)
    one, many = run(name, 8, flags, 3), run(name, 300, flags, 3)
    assert one['ncon'].min() > 0
    for k in FIELDS:
        np.testing.assert_array_equal(many[k][:8], one[k], err_msg=k)
        np.testing.assert_array_equal(many[k][288:296], one[k], err_msg=k)
    a, b = run(name, 8, flags, 1), run(name, 8, 0, 1)
    assert np.array_equal(a['ncon'], b['ncon']) and np.array_equal(a['contact_geom'], b['contact_geom'])
    assert np.abs(a['qpos'] - b['qpos']).max() < 1e-6
    for k in ('qvel', 'qacc', 'M', 'qfrc_bias', 'osc_tau'):
        assert rel_err(a[k], b[k]) < 1e-4, k
