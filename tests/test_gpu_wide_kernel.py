"""The kernels with several waves per world against the one-wave kernel, bit for bit.

The launch picks four waves per world up to four worlds per CU, two up to eight, one beyond, where the
CU's LDS holds their windows, and widens the window up to sixteen worlds per CU.  The same worlds are
run alone and repeated through batches on both sides of each limit (from the device's CU count); each
must end with the same bits whatever kernel and window stepped it: contacts and their order, rows,
solver and controller state, observations.  Scenes: pyramidal and elliptic cones, hulls, MPR, parked
bodies, dense clutter (the most contacts, and a base window without contact staging), and a LIBERO task
whose pair table and candidates span several parts and rounds; then a contact array too small for the
scene, and masked passes.
"""
from pathlib import Path

import numpy as np
import pytest

from libero_hip import native, observations, scene as S, scene_io
from libero_hip.model import Model

pytestmark = pytest.mark.gpu

FIELDS = ('time', 'qpos', 'qvel', 'qacc', 'qacc_warmstart', 'qfrc_constraint', 'qfrc_bias', 'M', 'ctrl', 'osc_tau',
          'osc_goal_pos', 'osc_goal_rot', 'osc_gripper', 'cfrc_ext', 'cfrc_int', 'xpos', 'subtree_com', 'ncon', 'nefc',
          'contact_pos', 'contact_frame', 'contact_geom', 'efc_force', 'efc_type', 'solver_niter', 'overflow', 'nstep',
          'stat_sums')
NARROWPHASE = 1 << 3          # MX_OVERFLOW_NARROWPHASE


def run(sc, nworld, substeps):
    import torch
    base = sc.init_qpos.shape[0]
    pick = np.arange(nworld) % base
    m = Model(sc)
    d = native.DeviceData(native.DeviceModel(m), nworld)
    rng = np.random.default_rng(3)
    qvel = np.zeros((base, m.nv))
    qvel[:, :7] = rng.uniform(-0.4, 0.4, (base, 7))
    d['qpos'].copy_(torch.from_numpy(sc.init_qpos[pick]))
    d['qvel'].copy_(torch.from_numpy(qvel[pick]))
    d['osc_gains'].copy_(torch.from_numpy(np.tile(np.r_[sc.osc['kp'], sc.osc['kd']], (nworld, 1))))
    d['osc_q0'].copy_(torch.from_numpy(np.tile(np.asarray(sc.osc['q0'], float), (nworld, 1))))
    d['osc_action'].copy_(torch.from_numpy(rng.uniform(-1, 1, (base, 7))[pick]))
    active = np.ones((base, m.nbody), np.int32) if m.body_active is None else m.body_active
    d['body_active'].copy_(torch.from_numpy(active[pick]))
    obs = observations.DeviceObservations(observations.default_plan(m), m, nworld)
    d.forward(None, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL)
    obs.control_step(d, substeps, native.FLAG_POLICY_FIRST)
    torch.cuda.synchronize()
    return {**{k: d[k].cpu().numpy() for k in FIELDS}, 'observed': obs.observed.cpu().numpy()}


def batches():
    """Batch sizes on both sides of four, eight and sixteen worlds per CU."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return 4 * cus, 4 * cus + 1, 8 * cus, 8 * cus + 1, 16 * cus + 1


def scene(name):
    if name.startswith('libero'):
        sc = scene_io.load(Path(__file__).resolve().parent / 'golden' / (name + '.json'))
        a = Model(sc).arrays
        free = [int(q) for q, t in zip(a['jnt_qposadr'], a['jnt_type']) if t == S.FREE]
        for q, landed in zip(free, (0.0315, 0.0325, 0.0284, 0.0318, 0.0005)):   # onto their supports
            sc.init_qpos[:, q + 2] -= landed
    else:
        sc = S.make_scene(name[:2], 16, seed=4)
        sc.options.mpr = name.endswith('mpr')
        for k in range((sc.init_qpos.shape[1] - 9) // 7):      # from the drop height onto the table
            sc.init_qpos[:, 11 + 7 * k] -= np.where(sc.init_qpos[:, 11 + 7 * k] > 0, 0.0051, 0.0)
    return sc


def check_batches(name, sc):
    want = None
    for nworld in (16,) + batches():
        print('case', name, nworld, flush=True)
        out = run(sc, nworld, 8)
        first = {k: v[:16] for k, v in out.items()}
        if want is None:
            want = first
            assert want['ncon'].max() > 0
        for k in want:
            np.testing.assert_array_equal(first[k], want[k], err_msg='%s %d' % (k, nworld))
            for at in (16 * ((nworld - 1) // 16), 16 * (nworld // 32)):
                n = min(16, nworld - at)
                np.testing.assert_array_equal(out[k][at:at + n], want[k][:n], err_msg='%s %d' % (k, nworld))
    return want


@pytest.mark.parametrize('name', ['c1', 'c3', 'c3-mpr', 'c4', 'c5', 'libero_spatial_bowl_plate'])
def test_waves_per_world_do_not_change_results(gpu_available, name):
    check_batches(name, scene(name))


@pytest.mark.parametrize('name', ['c3', 'c4', 'libero_spatial_bowl_plate'])
def test_contacts_beyond_the_array(gpu_available, name):
    """The contacts that are kept are the first in candidate order, also where the array ends within a
    wave's share, and every kernel flags the loss (two thirds of what the scene needs)."""
    sc = scene(name)
    sc.options.nconmax = nconmax = int(run(sc, 16, 8)['ncon'].max()) * 2 // 3
    want = check_batches(name, sc)
    assert (want['ncon'] == nconmax).any() and ((want['overflow'] & NARROWPHASE) != 0).any()


@pytest.mark.parametrize('name', ['c5', 'libero_spatial_bowl_plate'])
def test_masked_pass(gpu_available, name):
    """A masked forward pass: the selected worlds as in a pass of sixteen, the others untouched."""
    import torch
    sc = scene(name)
    m = Model(sc)
    active = np.ones((16, m.nbody), np.int32) if m.body_active is None else m.body_active
    want = None
    for nworld in (16,) + batches():
        print('case', name, nworld, flush=True)
        pick = np.arange(nworld) % 16
        chosen = np.random.default_rng(nworld).random(nworld) < 0.5
        d = native.DeviceData(native.DeviceModel(m), nworld)
        for k, v in dict(qpos=sc.init_qpos, body_active=active).items():
            d[k].copy_(torch.from_numpy(np.ascontiguousarray(v[pick])))
        before = {k: d[k].cpu().numpy() for k in FIELDS}
        mask = None if nworld == 16 else torch.from_numpy(chosen.astype(np.int32)).to(d['qpos'].device)
        d.forward(mask, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL)
        torch.cuda.synchronize()
        out = {k: d[k].cpu().numpy() for k in FIELDS}
        if want is None:
            want = out
            assert want['ncon'].max() > 0
            continue
        for k in FIELDS:
            np.testing.assert_array_equal(out[k][chosen], want[k][pick[chosen]], err_msg='%s %d' % (k, nworld))
            np.testing.assert_array_equal(out[k][~chosen], before[k][~chosen], err_msg='%s %d' % (k, nworld))
