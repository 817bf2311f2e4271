"""A quotient formed with a shared reciprocal of its divisor has the bits of a
division (needs an MI355X): pixel coordinates of a detector centred on pixel 0
are local coordinates over the pixel size and nothing else, so FP64 traces have
to give numpy's quotients bit for bit, over random mantissas, 280 decades of
numerators and 20 of divisors, zeros of both signs among them.  Rays along x
keep their y and z."""
import numpy as np
import pytest

import marxs_amd as mx
from tests.helpers import gpu_trace

pytestmark = pytest.mark.gpu

N = 60000


def _rays(rng, half):
    yz = rng.uniform(-1, 1, (N, 2)) * half * 10. ** -np.where(rng.random((N, 2)) < 0.5, rng.uniform(0, 3, (N, 2)),
                                                              rng.uniform(0, 270, (N, 2)))
    yz[:50] = 0.
    yz[50:100] = -0.
    pol = np.zeros((N, 3))
    pol[:, 2] = 1.
    return {'pos': np.column_stack([np.full(N, 5.), yz]), 'dir': np.tile([-1., 0., 0.], (N, 1)), 'pol': pol,
            'energy': np.ones(N), 'prob': np.ones(N)}


@pytest.mark.parametrize('seed', range(6))
@pytest.mark.parametrize('pair', [False, True])
def test_flat_detector(gpu, seed, pair):
    rng = np.random.default_rng(seed)
    half = 10. ** rng.uniform(-10, 10)
    size = half * rng.uniform(1, 2) * 10. ** -rng.uniform(0, 7)
    args = {'pixsize': size, 'zoom': [1., half, half], 'ignore_pixel_warning': True}
    # the second of a pair lies beside the beam
    det = mx.Parallel(elem_class=mx.FlatDetector, elem_args=args, id_col='CCD',
                      elem_pos={'position': [[0, 0, 0], [0, 9 * half, 9 * half]][:1 + pair]})
    for e in det.elements:
        e.centerpix = [0, 0]
    ph = _rays(rng, half)
    got, _ = gpu_trace(mx.Sequence(elements=[det]), ph, np.zeros((1, N)))
    assert np.all(got['CCD'] == 0) and np.array_equal(got['det_x'], ph['pos'][:, 1])
    for a, b in (('detpix_x', 'det_x'), ('detpix_y', 'det_y')):
        assert np.array_equal((got[b] / size).view(np.int64), got[a].view(np.int64))


@pytest.mark.parametrize('seed', range(6))
def test_tube(gpu, seed):
    rng = np.random.default_rng(100 + seed)
    size = rng.uniform(1, 2) * 10. ** -rng.uniform(-9, 9)
    tube = mx.CircularDetector(pixsize=size, zoom=[3., 3., 2.])
    ph = _rays(rng, 1.9)
    got, _ = gpu_trace(mx.Sequence(elements=[tube]), ph, np.zeros((1, N)))
    assert np.all(np.isfinite(got['det_y']))
    assert np.array_equal((got['det_y'] / size).view(np.int64), got['detpix_y'].view(np.int64))
    assert np.array_equal((got['det_phi'] * 3. / size).view(np.int64), got['detpix_x'].view(np.int64))
