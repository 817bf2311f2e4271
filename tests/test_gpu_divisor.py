"""Quotients that share a divisor (needs an MI355X): a direction scaled by a
power of two has the same unit vector, so an FP64 trace of it gives the same
bits; components that are zero or tiny stay what the oracle's division gives."""
import numpy as np
import pytest

from marxs_amd import configs
from marxs_amd.tracer import CompiledInstrument
from tests.helpers import compare, gpu_trace, make_inputs, near_pixel_boundary, oracle_trace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('exponent', [-400, -1, 1, 400])
def test_scaled_directions(gpu, exponent):
    inst, _ = configs.cat_rowland_instrument(200)
    ci = CompiledInstrument(inst)
    n = 2051
    ph, u = make_inputs(n, 3, ci.n_uniform_slots)
    # zero, negative zero and tiny components beside ordinary ones
    ph['dir'][:, 1:] = 0.
    ph['dir'][: n // 4, 1] = -0.
    ph['dir'][n // 4: n // 2, 2] = 1e-250
    ph['dir'][n // 2:, 1] = np.linspace(-1e-4, 1e-4, n - n // 2)
    ph['dir'] /= np.linalg.norm(ph['dir'], axis=1)[:, None]
    a, _ = gpu_trace(ci, ph, u)
    compare(oracle_trace(inst, ph, u), a, rtol=1e-9, near=near_pixel_boundary(a))
    b, _ = gpu_trace(ci, {**ph, 'dir': ph['dir'] * 2. ** exponent}, u)
    for k in a:
        if k != 'prob' and not k.startswith('aper'):    # the projected area scales with the direction
            assert np.array_equal(a[k], b[k], equal_nan=a[k].dtype.kind == 'f'), k
