"""The LDS route's two-wave kernel: the same worlds bit for bit at any place and size of a batch, on
both precisions, and to FP32 rounding the workspace route's result (one substep: positions 1e-6,
velocities and accelerations by their scale 1e-4, the parity bar of the two routes).  Models small
enough for three or four worlds in a CU's LDS take one wave per world in batches that fill them so:
the same bits on either side."""
import numpy as np
import pytest

from helpers import rel_err
from test_gpu_wide_kernel import FIELDS
from libero_hip import native, scene as S
from libero_hip.model import Model

pytestmark = pytest.mark.gpu


def run(name, nworld, flags, substeps, nobjects=None, nconmax=64):
    import torch
    sc = S.make_scene(name, 8, seed=4, nobjects=nobjects)
    sc.options.nconmax = nconmax
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


@pytest.mark.parametrize('route,nobjects', [('lds', 1), ('fp64', 0)])
def test_one_wave_and_two_waves_agree(gpu_available, route, nobjects):
    import torch
    flags = native.FLAG_LDS if route == 'lds' else native.FLAG_FP64
    sc = S.make_scene('c1', 1, nobjects=nobjects)
    sc.options.nconmax = 24
    dm = native.DeviceModel(Model(sc))
    assert (dm.lds_bytes() if route == 'lds' else dm.lds_bytes_fp64()) <= 163840 // 3     # three worlds per CU at least
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    one = run('c1', 8, flags, 6, nobjects, 24)
    assert one['nefc'].max() > 0 or nobjects == 0
    for nworld in (2 * cus, 2 * cus + 1, 3 * cus, 6 * cus + 3):      # two waves; one wave
        print('case', route, nworld, flush=True)
        many = run('c1', nworld, flags, 6, nobjects, 24)
        for k in FIELDS:
            pick = np.arange(nworld) % 8
            np.testing.assert_array_equal(many[k], one[k][pick], err_msg='%s %d' % (k, nworld))
