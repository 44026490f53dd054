"""mx_osc packs eight worlds into a wavefront: batches around whole waves, with worlds in one wave that
take different ways through the controller, each against the FP64 oracle on the same inputs; and an
infinite joint state, which must reach the torques as it does there."""
import numpy as np
import pytest

from tests.helpers import rel_err
from tests.test_gpu_smooth_parity import _np, _pair, six_joint_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('joints,nworld,uncouple,policy', [
    (7, 1, 1, True), (7, 7, 1, True), (7, 8, 0, True), (7, 9, 1, False), (7, 67, 1, True), (6, 13, 0, True)])
def test_osc_groups(gpu_available, joints, nworld, uncouple, policy):
    """Worlds by w % 5: 0 and 4 regular (4 without a rotation in its action), 1 a mass matrix that is not
    positive definite (the error, and nothing else written), 2 two equal Jacobian rows (the pseudo-inverse
    fallback, rank 5 and 2), 3 in error before the call (nothing written).  tau is compared to 1e-9: the
    operations are 64-bit and A's condition reaches 1e6 on such draws (a mean one's is 1e2 to 1e3), so
    rounding is below 1e6 x 2^-53 = 1e-10."""
    import torch
    from libero_hip import scene as S, native
    from oracle import oracle as O
    sc = six_joint_scene(nworld) if joints == 6 else S.make_scene('c2', nworld, seed=0)
    sc.osc = dict(sc.osc, uncouple=uncouple)
    m, dd, _ = _pair('c2', nworld, scene=sc)
    n = m.osc_ndof
    assert n == joints and m.osc_uncouple == uncouple
    rng = np.random.default_rng(100 * joints + nworld)
    kind = np.arange(nworld) % 5
    L = rng.normal(size=(nworld, n, n)) * 0.2 + np.eye(n)
    mass = L @ L.transpose(0, 2, 1)
    mass[kind == 1, 2, 2] = -1.0
    jac = rng.normal(size=(nworld, 6, n))
    if n == 6:   # square: keep A's condition bounded
        jac += 3.0 * np.eye(6)
    jac[kind == 2, 1] = jac[kind == 2, 0]
    from scipy.spatial.transform import Rotation
    turn = lambda: Rotation.from_rotvec(rng.normal(size=(nworld, 3))).as_matrix().reshape(nworld, 9)  # noqa: E731
    acts = rng.uniform(-1.2, 1.2, (nworld, 7))
    acts[kind == 4, 3:6] = 0.0
    fields = dict(osc_mass=mass.reshape(nworld, -1), osc_jac=jac.reshape(nworld, -1), osc_q=rng.normal(size=(nworld, n)),
                  osc_qvel=rng.normal(size=(nworld, n)), osc_bias=rng.normal(size=(nworld, n)),
                  osc_ee_pos=rng.normal(size=(nworld, 3)), osc_ee_rot=turn(), osc_ee_vel=rng.normal(size=(nworld, 6)),
                  osc_goal_pos=rng.normal(size=(nworld, 3)), osc_goal_rot=turn(),
                  osc_gripper=rng.uniform(-1, 1, (nworld, 2)), osc_action=acts,
                  osc_error=np.where(kind == 3, 4, 0)[:, None], osc_rank=np.full((nworld, 3), -7),
                  ctrl=rng.normal(size=(nworld, m.nu)), osc_tau=rng.normal(size=(nworld, n)))
    for k, v in fields.items():
        dd[k].copy_(torch.from_numpy(np.ascontiguousarray(v)).reshape(dd[k].shape))
    before = {k: _np(dd[k]).reshape(nworld, -1).copy() for k in fields}
    dd.osc(native.FLAG_POLICY_FIRST if policy else 0)
    torch.cuda.synchronize()
    after = {k: _np(dd[k]).reshape(nworld, -1) for k in fields}
    crange = m.arrays['actuator_ctrlrange'][m.arrays['osc_actuator']].reshape(-1)
    for w in range(nworld):
        if kind[w] == 3:
            for k in fields:
                assert np.array_equal(after[k][w], before[k][w]), (w, k)
            continue
        inp = {k: before['osc_' + k][w] for k in ('mass', 'jac', 'q', 'qvel', 'bias', 'ee_pos', 'ee_rot', 'ee_vel')}
        err, tau, ctrl, rank, gp, gr, gg = O.osc(inp, acts[w], _np(dd['osc_gains'])[w], _np(dd['osc_q0'])[w], crange,
                                                 before['osc_goal_pos'][w], before['osc_goal_rot'][w],
                                                 before['osc_gripper'][w], policy=policy, uncouple=uncouple,
                                                 speed=float(np.float32(m.osc_gripper_speed)))
        assert after['osc_error'][w, 0] == err, w
        if kind[w] == 1:
            assert err != 0
            for k in fields:
                assert k == 'osc_error' or np.array_equal(after[k][w], before[k][w]), (w, k)
            continue
        assert np.array_equal(after['osc_rank'][w], rank), w
        assert list(rank) == ([5, 2, 3] if kind[w] == 2 else [6, 3, 3])
        assert rel_err(after['osc_tau'][w], tau) < 1e-9, w
        np.testing.assert_allclose(after['osc_goal_pos'][w], gp, rtol=0, atol=1e-12)
        np.testing.assert_allclose(after['osc_goal_rot'][w], gr, rtol=0, atol=1e-12)
        np.testing.assert_array_equal(after['osc_gripper'][w], gg)
        np.testing.assert_allclose(after['ctrl'][w, m.arrays['osc_actuator']], ctrl, rtol=1e-6, atol=1e-6)
        others = np.setdiff1d(np.arange(m.nu), m.arrays['osc_actuator'])
        assert np.array_equal(after['ctrl'][w, others], before['ctrl'][w, others])


def test_infinite_joint_state(gpu_available):
    """An infinite first joint velocity: the posture torques are infinite, and a torque is infinite or NaN
    as its nullspace terms' signs agree or not.  With seven joints a wave's eighth lane holds no joint."""
    import torch
    from libero_hip import native, scene as S
    from oracle import oracle as O
    nworld = 200
    m, dd, _ = _pair('c2', nworld, scene=S.make_scene('c2', nworld, seed=0))
    n = m.osc_ndof
    rng = np.random.default_rng(71)
    L = rng.normal(size=(nworld, n, n)) * 0.2 + np.eye(n)
    qvel = rng.normal(size=(nworld, n))
    qvel[:, 0] = np.where(np.arange(nworld) % 2, np.inf, -np.inf)
    fields = dict(osc_mass=(L @ L.transpose(0, 2, 1)).reshape(nworld, -1), osc_jac=rng.normal(size=(nworld, 6 * n)),
                  osc_q=rng.normal(size=(nworld, n)), osc_qvel=qvel, osc_bias=rng.normal(size=(nworld, n)),
                  osc_ee_pos=rng.normal(size=(nworld, 3)), osc_ee_rot=np.tile(np.eye(3).reshape(9), (nworld, 1)),
                  osc_ee_vel=rng.normal(size=(nworld, 6)), osc_goal_pos=rng.normal(size=(nworld, 3)),
                  osc_goal_rot=np.tile(np.eye(3).reshape(9), (nworld, 1)), osc_action=rng.uniform(-1, 1, (nworld, 7)))
    for k, v in fields.items():
        dd[k].copy_(torch.from_numpy(np.ascontiguousarray(v)).reshape(dd[k].shape))
    inp = {k: _np(dd['osc_' + k]).reshape(nworld, -1) for k in ('mass', 'jac', 'q', 'qvel', 'bias', 'ee_pos', 'ee_rot', 'ee_vel')}
    grip = _np(dd['osc_gripper']).copy()
    dd.osc(0)
    torch.cuda.synchronize()
    tau, ctrl = _np(dd['osc_tau']).reshape(nworld, -1), _np(dd['ctrl']).reshape(nworld, -1)
    acts = m.arrays['osc_actuator']
    infinite = 0
    for w in range(nworld):
        _, want, wctrl, *_ = O.osc({k: v[w] for k, v in inp.items()}, fields['osc_action'][w], _np(dd['osc_gains'])[w],
                                   _np(dd['osc_q0'])[w], m.arrays['actuator_ctrlrange'][acts].reshape(-1),
                                   fields['osc_goal_pos'][w], fields['osc_goal_rot'][w], grip[w], policy=False,
                                   uncouple=m.osc_uncouple, speed=float(np.float32(m.osc_gripper_speed)))
        infinite += np.isinf(want).sum()
        assert not np.isfinite(want).any()
        np.testing.assert_array_equal(tau[w], want)
        np.testing.assert_array_equal(ctrl[w, acts[:n]], wctrl[:n].astype(np.float32))
    assert infinite > 20


@pytest.mark.parametrize('config,nworld', [('c2', 21), ('c3', 21)])
def test_osc_is_the_step_kernels_controller(gpu_available, config, nworld):
    """mx_osc on the inputs that a control step's substep published gives that substep's torques, goal,
    gripper and controls bit for bit (both kernels run the same 64-bit operations in the same order)."""
    import torch
    from libero_hip import native, scene as S
    from libero_hip.model import Model
    sc = S.make_scene(config, nworld, seed=2)
    m = Model(sc)
    d = native.DeviceData(native.DeviceModel(m), nworld)
    rng = np.random.default_rng(22)
    d['qpos'].copy_(torch.from_numpy(sc.init_qpos))
    d['qvel'][:, :7].copy_(torch.from_numpy(rng.uniform(-1, 1, (nworld, 7))))
    d['osc_gains'].copy_(torch.from_numpy(np.tile(np.r_[sc.osc['kp'], sc.osc['kd']], (nworld, 1))))
    d['osc_q0'].copy_(torch.from_numpy(np.tile(np.asarray(sc.osc['q0'], float), (nworld, 1))))
    d['osc_action'].copy_(torch.from_numpy(rng.uniform(-1, 1, (nworld, 7))))
    d['body_active'].fill_(1)
    d.forward(None, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL)
    before = {k: d[k].clone() for k in ('osc_goal_pos', 'osc_goal_rot', 'osc_gripper', 'ctrl')}
    d.control_step(1, native.FLAG_POLICY_FIRST)
    fields = ('osc_tau', 'osc_goal_pos', 'osc_goal_rot', 'osc_gripper', 'ctrl', 'osc_rank', 'osc_error')
    want = {k: d[k].clone() for k in fields}
    for k, v in before.items():
        d[k].copy_(v)
    d['osc_tau'].zero_()
    d.osc(native.FLAG_POLICY_FIRST)
    torch.cuda.synchronize()
    assert want['osc_tau'].abs().max() > 0 and not torch.equal(want['osc_goal_rot'], before['osc_goal_rot'])
    for k in fields:
        assert torch.equal(d[k], want[k]), k
