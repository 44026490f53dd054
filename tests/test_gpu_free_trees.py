"""Trees without a constraint row stay out of the Newton blocks; their part of the joint solve's steps
is followed by three sums and the product of 1 - alpha.  The oracle solves all trees together: every
tree's accelerations and the iteration counts of most worlds must be its (the parity bar 1e-4), and
the free trees end within it of qacc_smooth.

The arm free, held by a joint limit, or with dof friction rows; parked objects; both routes.
"""
import numpy as np
import pytest

from helpers import rel_err
from libero_hip import native, scene as S
from test_gpu_contact_parity import _settled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('config,arm', [('c1', 'free'), ('c3', 'free'), ('c3', 'limit'), ('c3', 'friction'),
                                        ('c5', 'free')])
@pytest.mark.parametrize('route', ['workspace', 'lds'])
def test_free_trees_follow_the_joint_solve(gpu_available, config, arm, route):
    import torch
    nworld = 16
    sc = S.make_scene(config, nworld, seed=6)
    if arm == 'friction':
        sc.bodies[3].joints[0].frictionloss = 0.2
    if arm == 'limit':
        sc.init_qpos[:, 4] = 2.905           # beyond the joint's upper limit
    print('case', config, arm, route, flush=True)
    m, dd, od, acts = _settled(config, nworld, settle=1 if arm == 'limit' else 2, seed=6, scene=sc,
                               workspace=None if route == 'workspace' else False)
    dd['osc_action'].copy_(torch.from_numpy(acts[0]))
    od['osc_action'][:] = acts[0]
    dd.control_step(1, native.FLAG_POLICY_FIRST)
    od.control_step(1, native.FLAG_POLICY_FIRST)
    torch.cuda.synchronize()
    g = {k: dd[k].cpu().numpy() for k in ('qacc', 'qacc_smooth', 'ncon', 'nefc', 'contact_geom', 'efc_type', 'efc_id')}
    a = {k: np.asarray(v).reshape(-1) for k, v in m.arrays.items()}
    free = 0
    for w in range(nworld):
        touched = set()
        for c in range(g['ncon'][w, 0]):
            for q in (0, 1):
                touched.add(int(a['body_treeid'][a['geom_body'][g['contact_geom'][w, 2 * c + q]]]))
        for r in range(g['nefc'][w, 0]):
            kind, row = g['efc_type'][w, r], g['efc_id'][w, r]
            if kind < 5:
                touched.add(int(a['dof_treeid'][row if kind == 1 else a['jnt_dofadr'][row]]))
        off = np.array([int(t) not in touched for t in a['dof_treeid']])
        free += off.sum()
        if g['nefc'][w, 0]:
            scale = np.abs(od['qacc'][w]).max()
            assert np.abs(g['qacc'][w, off] - g['qacc_smooth'][w, off]).max(initial=0.0) < 1e-4 * scale
            assert np.abs(g['qacc'][w, off] - od['qacc'][w, off]).max(initial=0.0) < 1e-5 * scale
    assert (free > 0) if arm == 'free' else free < nworld * 9 or config == 'c5'
    assert rel_err(g['qacc'], od['qacc']) < 1e-4
    niter = dd['solver_niter'].cpu().numpy()[:, 0]
    assert (niter == od['solver_niter'].reshape(-1)).mean() > 0.5
