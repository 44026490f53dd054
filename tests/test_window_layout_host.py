"""The workspace route's LDS window, from its layout code compiled for the host.

* The window of every scene, which the Newton solve lays itself out in and so rounds by, is that of an
  EPA polytope of the reference's 10 + 2 it vertices, except where only the smaller polytope lets
  sixteen worlds share a CU;
* a launch that widens it (more row-group EPA blocks, several waves per world) stays inside the CU's
  LDS, leaves the Newton solve its layout, and keeps the parts apart that waves write at once.

And the LDS route's choice of one or two waves per world, which must not cost a batch residency.
"""
import ctypes as ct
import subprocess
from pathlib import Path

import pytest

from libero_hip import layout, native, scene as S, scene_io
from libero_hip.model import Model

ROOT = Path(__file__).resolve().parents[1]
NAMES = ('win', 'nwin', 'epa', 'epa_req', 'epa_vc', 'epa_fc', 'gpose', 'meshw', 'stage', 'epa_ng', 'epa_gw', 'swin', 'ewin',
         'ewords')
SOURCE = '''
#include "%s"
extern "C" int window(const MxModel* m, int nworld, int ncu, int waves, int* out) {
  using namespace mx_slab;
  Layout L = make_layout(*m);
  const bool fits = nworld == 0 || widen_window(L, *m, nworld, ncu, waves);
  const int v[] = {%s};
  for (int i = 0; i < %d; ++i) out[i] = v[i];
  return fits;
}
extern "C" int polytope_words(int vertices, int faces) { return mx_slab::cvx::poly_words(vertices, faces); }
'''
WAVES_SOURCE = '''
#include "%s"
extern "C" int two_waves(int nworld, int bytes, int ncu) { return mx_f64::two_waves(nworld, bytes, ncu); }
'''
REQUEST, CLIP, SCALARS, COUNTS, CUS = 48, 88, 48, 16, 256
SCENES = ['c1', 'c3', 'c4', 'c5', 'libero_spatial_bowl_plate', 'libero_goal_wine_rack']


def compiled(at, source):
    """The host half of a HIP source alone: an empty device image, nothing launched."""
    import build
    (at / 'source.hip').write_text(source)
    subprocess.run([build.hipcc(), '--offload-arch=gfx950', '--offload-host-only', '-fuse-cuid=none', '-O0', '-std=c++17',
                    '-fPIC', '-shared', '-o', str(at / 'source.so'), str(at / 'source.hip'),
                    '-Wl,--defsym,__hip_fatbin=0'], check=True)
    return ct.CDLL(str(at / 'source.so'))


@pytest.fixture(scope='module')
def lib(tmp_path_factory):
    slab = ROOT / 'gpu-libero_amd' / 'csrc' / 'mx_step_slab.hip'
    return compiled(tmp_path_factory.mktemp('window'), SOURCE % (slab, ', '.join('L.' + n for n in NAMES), len(NAMES)))


def model(name):
    sc = S.make_scene(name, 2, seed=0) if len(name) == 2 else scene_io.load(ROOT / 'tests' / 'golden' / (name + '.json'))
    m, s = Model(sc), native.MxModel()
    for k, v in layout.model_scalars(m).items():
        setattr(s, k, v)
    return m, s


def window(lib, s, nworld=0, waves=1):
    out = (ct.c_int * len(NAMES))()
    fits = lib.window(ct.byref(s), nworld, CUS, waves, out)
    return bool(fits), dict(zip(NAMES, out))


@pytest.mark.parametrize('name', SCENES)
def test_window_of_a_scene(lib, name):
    m, s = model(name)
    _, w = window(lib, s)
    collision = lambda vertices: (-(-(-(-lib.polytope_words(vertices, w['epa_fc']) // 4) * 4 + REQUEST + CLIP  # noqa: E731
                                      + 21 * m.ngeom) // 4) * 4 + 4 * m.nmeshvert + 3) // 4 * 4
    full, small = collision(10 + 2 * m.epa_iterations), collision(6 + m.epa_iterations)
    sixteen = layout.LDS_BUDGET // 16 // 4 - SCALARS
    assert w['win'] == w['nwin'] == max(sixteen, small if full > sixteen >= small else full)
    assert (full > sixteen >= small) == (name == 'c4')
    assert w['epa_vc'] >= 5 + m.epa_iterations


@pytest.mark.parametrize('name', SCENES)
@pytest.mark.parametrize('waves', [1, 2, 4])
def test_widened_window(lib, name, waves):
    m, s = model(name)
    _, base = window(lib, s)
    taken = 0
    for per_cu in range(1, 17):
        for nworld in (CUS * (per_cu - 1) + 1, CUS * per_cu):
            fits, w = window(lib, s, nworld, waves)
            if not fits:
                assert w == base
                continue
            taken += 1
            assert w['nwin'] == base['nwin'] <= w['win']
            nbytes = 4 * (w['win'] + SCALARS + (COUNTS if waves > 1 else 0))
            assert per_cu * (-(-nbytes // 1280) * 1280) <= layout.LDS_BUDGET
            # a wave's block: the polytope with its request, the row groups, the staging; then the records
            assert w['epa_req'] >= lib.polytope_words(w['epa_vc'], w['epa_fc'])
            assert w['gpose'] >= w['epa_req'] + REQUEST + CLIP and w['gpose'] >= w['epa_ng'] * w['epa_gw']
            assert w['stage'] == -1 or w['gpose'] >= 18 * 64 + 8 * m.nconmax
            assert w['gpose'] % 4 == 0 and w['meshw'] >= w['gpose'] + 21 * m.ngeom
            first = w['ewin'] if waves > 1 else w['win']
            assert w['meshw'] + 4 * m.nmeshvert <= first and w['nwin'] <= first
            if waves > 1:
                on = m.osc_ndof
                smooth = max(23 * m.nbody + 6 * m.nv, 16 * m.nbody + 6 * m.njnt, 2 * m.nu + m.nv,
                             2 * (2 * on * on + 12 * on + 36), 2 * (m.nM + m.nMdamp) if 2 * (m.nM + m.nMdamp) <= w['nwin'] else 0)
                assert w['ewords'] == w['gpose'] and w['swin'] >= w['ewin'] + (waves - 2) * w['ewords']
                assert w['swin'] + smooth <= w['win'] and w['ewin'] % 4 == w['swin'] % 2 == 0
    assert taken > 0


def test_lds_route_waves(tmp_path):
    """Two waves per world exactly where one wave per world would take as many rounds of resident
    worlds (a CU holds as many as its LDS, four of one wave or two of two)."""
    lib = compiled(tmp_path, WAVES_SOURCE % (ROOT / 'gpu-libero_amd' / 'csrc' / 'mx_step_f64.hip'))
    for nbytes in (20000, 40240, 48976, 50720, 58048, 69104, 85136, 163840):
        fit = layout.LDS_BUDGET // nbytes
        for nworld in (1, 16, CUS, CUS + 1, 2 * CUS, 2 * CUS + 1, 3 * CUS, 4 * CUS, 4 * CUS + 1, 8192, 16384):
            rounds = lambda most: -(-nworld // (CUS * min(fit, most)))  # noqa: E731
            assert bool(lib.two_waves(nworld, nbytes, CUS)) == (rounds(2) <= rounds(4)), (nbytes, nworld)
            assert fit > 2 or lib.two_waves(nworld, nbytes, CUS)
