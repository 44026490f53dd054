"""The broadphase's batched filter of the pair table against the oracle's contacts.

Sphere clusters on several free bodies give pair tables from below one round of 64 pairs (the counts
are printed) to several batches of 256 with a remainder in each wave's part, with margins and gaps, under
both margin rules, and with a parked body; a batch of more than eight worlds per CU runs the one-wave
kernel, which filters the whole table in one call.  Sphere contacts are closed forms, so the contacts' geom pairs and order are those of the
oracle exactly, and every pair within its threshold must be there: a pair the filter lost is missing.
Positions agree to 1e-5 m (FP32 rounding of poses of order 1 m and of normals of centimetre offsets).
"""
import numpy as np
import pytest

from helpers import make_oracle
from libero_hip import native, scene as S
from libero_hip.model import Model

pytestmark = pytest.mark.gpu


def cluster_scene(nbody, per_body, nworld, seed, mpr, parked, margins=(0.0, 0.002), gaps=(0.0, 0.001)):
    rng = np.random.default_rng(seed)
    arm, actuators, osc, q_ready = S._arm()
    bodies = [S._world(table=False)] + arm
    for k in range(nbody):
        b = S.Body('cluster%d' % k, 0, mass=0.3, inertia=(1e-4,) * 3)
        b.joints.append(S.Joint(S.FREE))
        for _ in range(per_body):
            b.geoms.append(S.Geom(S.SPHERE, size=(float(rng.uniform(0.005, 0.02)), 0.0, 0.0), condim=1,
                                  pos=tuple(float(x) for x in rng.uniform(-0.05, 0.05, 3)),
                                  margin=float(rng.choice(margins)), gap=float(rng.choice(gaps))))
        bodies.append(b)
    opts = S.Options()
    opts.nconmax, opts.mpr = 256, mpr
    qpos = np.zeros((nworld, 9 + 7 * nbody))
    qpos[:, :7] = q_ready
    qpos[:, 7:9] = 0.02
    for k in range(nbody):
        q = rng.normal(size=(nworld, 4))
        qpos[:, 9 + 7 * k:12 + 7 * k] = rng.uniform((1.2, -0.06, 0.03), (1.32, 0.06, 0.12), (nworld, 3))
        qpos[:, 12 + 7 * k:16 + 7 * k] = q / np.linalg.norm(q, axis=1, keepdims=True)
    active = None
    if parked:
        active = np.ones((nworld, len(bodies)), np.int32)
        active[::2, -1] = 0
    return S.Scene(name='clusters', bodies=bodies, actuators=actuators, options=opts, nworld=nworld, substeps=25,
                   osc=osc, init_qpos=qpos, init_qvel=np.zeros((nworld, 9 + 6 * nbody)), body_active=active, seed=seed)


@pytest.mark.parametrize('nbody,per_body,mpr,parked',
                         [(1, 1, False, False), (2, 3, False, True), (3, 4, True, False), (4, 5, False, True),
                          (5, 7, True, True), (7, 9, False, True), (7, 9, True, False)])
def test_batched_filter_keeps_every_pair(gpu_available, nbody, per_body, mpr, parked):
    compare(cluster_scene(nbody, per_body, 32, 10 * nbody + per_body, mpr, parked))


def test_whole_table_in_one_call(gpu_available):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    compare(cluster_scene(7, 9, 32, 5, False, True), 8 * cus + 32)


@pytest.mark.parametrize('mpr', [False, True])
def test_negative_margins_and_gaps(gpu_available, mpr):
    """A margin below minus a sphere's radius, and a pair whose threshold is the larger of a negative
    margin and zero: no pair is lost, and no sphere is taken for a plane."""
    compare(cluster_scene(5, 6, 32, 77, mpr, False, margins=(-0.03, -0.004, 0.0, 0.002), gaps=(-0.002, 0.0, 0.001)))


def compare(sc, nworld=None):
    """The scene's worlds, repeated to a batch of nworld, against the oracle."""
    import torch
    m = Model(sc)
    om, od = make_oracle(m, sc.nworld, fp32_model=True)
    nworld = nworld or sc.nworld
    pick = np.arange(nworld) % sc.nworld
    dd = native.DeviceData(native.DeviceModel(m), nworld)
    dd['qpos'].copy_(torch.from_numpy(sc.init_qpos[pick]))
    od['qpos'][:] = dd['qpos'].double().cpu().numpy()[:sc.nworld]
    dd['body_active'].copy_(torch.from_numpy(od['body_active'].astype(np.int32)[pick]))
    dd.forward(None, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL)
    od.forward(None, native.FLAG_BOOTSTRAP | native.FLAG_NO_CONTROL)
    torch.cuda.synchronize()
    ncon = dd['ncon'].cpu().numpy()[:, 0]
    print('pairs', m.arrays['pair_geom'].reshape(-1, 2).shape[0], 'contacts', ncon.sum(), flush=True)
    assert ncon.max() < m.nconmax and np.array_equal(ncon, od['ncon'].reshape(-1)[pick])
    geom, pos = dd['contact_geom'].cpu().numpy(), dd['contact_pos'].double().cpu().numpy()
    for w, c in enumerate(ncon):
        assert np.array_equal(geom[w, :2 * c], od['contact_geom'][pick[w], :2 * c])
        assert np.abs(pos[w, :3 * c] - od['contact_pos'][pick[w], :3 * c]).max(initial=0.0) < 1e-5
