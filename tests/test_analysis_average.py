"""The 1-d area-weighted average without masked arrays gives the masked
arrays' numbers, bit for bit."""
import numpy as np
import pytest

from marxs_amd.analysis import _average_R_Aeff_1d, average_R_Aeff


@pytest.mark.parametrize('n', [0, 1, 7, 8, 9, 14, 20, 130])
@pytest.mark.parametrize('bad', [0., 0.4, 1.])
@pytest.mark.parametrize('zero', [0., 1.])
def test_same_numbers(n, bad, zero):
    rng = np.random.default_rng(n)
    r, a = rng.lognormal(5, 2, n), rng.lognormal(0, 2, n)
    r[rng.random(n) < bad] = np.nan
    a[rng.random(n) < zero] = 0.
    r[n // 2:n // 2 + 1] = np.inf
    with np.errstate(all='ignore'):
        x, y = average_R_Aeff(r, a), _average_R_Aeff_1d(r, a)
    for p, q in zip(x, y):
        assert type(p) is type(q)
        assert p is q or np.array_equal(p, q, equal_nan=True)
