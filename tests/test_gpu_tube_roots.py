"""Tube stages where the nearer root fails a test the farther one passes, and
the facet frame behind facets whose ids the trace does or does not create
(needs an MI355X).  FP64 against the oracle: floats within 1e-9 relative (both
run the same formulas in float64), ids exact."""
import numpy as np
import pytest

import marxs_amd as mx
from marxs_amd import catgrating as CG
from marxs_amd import configs
from marxs_amd.geometry import Cylinder
from marxs_amd.scatter import RadialMirrorScatter
from tests.helpers import compare, gpu_trace, make_inputs, near_pixel_boundary, oracle_trace

pytestmark = pytest.mark.gpu


# azimuth limits around 0, across the wrap at pi, one that excludes the near
# root of most rays, and limits of more than a turn
@pytest.mark.parametrize('phi_lim', [[-1., 1.], [2.5, 4.], [-0.1, 0.1], [-9., -7.]])
@pytest.mark.parametrize('inside', [True, False])
def test_root_choice(gpu, phi_lim, inside):
    rng = np.random.default_rng(12)
    tube = mx.CircularDetector(pixsize=0.01, zoom=[3., 3., 1.5], position=[0.3, -0.2, 0.1],
                               geometry=Cylinder, phi_lim=phi_lim, id_col='tube', id_num=1)
    inst = mx.Sequence(elements=[tube])
    n = 4099
    d = rng.normal(size=(n, 3))
    pos = rng.uniform(-1, 1, (n, 3)) if inside else -10 * d / np.linalg.norm(d, axis=1)[:, None] + \
        rng.uniform(-2, 2, (n, 3))
    # rays along the axis (no root) and rays in the plane phi = 0
    d[:5] = [0, 0, 1]
    d[5:60, 1] = 0
    pos[5:60, 1] = -0.2
    d /= np.linalg.norm(d, axis=1)[:, None]
    pol = np.cross(d, rng.normal(size=(n, 3)))
    pol /= np.linalg.norm(pol, axis=1)[:, None]
    ph = {'pos': pos, 'dir': d, 'pol': pol, 'energy': np.ones(n), 'prob': np.ones(n)}
    u = np.zeros((1, n))
    ref = oracle_trace(inst, ph, u)
    got, _ = gpu_trace(inst, ph, u)
    assert 0 < np.isfinite(ref['det_phi']).sum() < n
    compare(ref, got, rtol=1e-9, near=near_pixel_boundary(ref))


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('frame_last', [False, True])
def test_facet_frame(gpu, precision, frame_last):
    """catsupportbars right behind the facets, and behind a detector (another
    id column is written in between)."""
    inst0, parts = configs.cat_rowland_instrument(200)
    rms = RadialMirrorScatter(inplanescatter=2e-5, perpplanescatter=4e-6, position=[12500., 0, 0],
                              zoom=[1, 700, 700])
    tail = [parts['ccds'], CG.catsupportbars] if frame_last else [CG.catsupportbars, parts['ccds']]
    inst = mx.Sequence(elements=[parts['aperture'], parts['lens'], rms, parts['gratings']] + tail)
    from marxs_amd.tracer import CompiledInstrument
    ci = CompiledInstrument(inst)
    ph, u = make_inputs(5003, 7, ci.n_uniform_slots)
    got, _ = gpu_trace(ci, ph, u, precision=precision)
    assert 0 < (got['facet'] < 0).sum() < 5003
    assert np.array_equal(got['prob'] == 0, got['facet'] < 0)
    if precision == 64:
        ref = oracle_trace(inst, ph, u)
        compare(ref, got, rtol=1e-9, near=near_pixel_boundary(ref))
