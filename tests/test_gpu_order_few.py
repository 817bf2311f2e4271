"""Sigma clipping of orders with few photons at a narrow sigma (needs an
MI355X), where the kept values end as a pair whose two values lie exactly one
standard deviation from their median: with the same quotients, squares and root
as numpy's both stay.  Counts equal numpy's; medians are values or means of two
and equal; mean and standard deviation of up to 70 values of size 1 differ by
less than 70 units of 1.1e-16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clip(x, sigma, rounds=5):
    for _ in range(rounds):
        n = x.size
        if n == 0:
            break
        med, sd = np.median(x), np.std(x)
        x = x[(x >= med - sigma * sd) & (x <= med + sigma * sd)]
        if x.size == n:
            break
    return x


@pytest.mark.parametrize('sizes', [(2, 2), (2, 9), (10, 70)])
@pytest.mark.parametrize('sigma', [1., 0.8, 3.])
def test_counts_of_few(gpu, sizes, sigma):
    import torch
    from marxs_amd import analysis
    rng = np.random.default_rng(int(10 * sigma) + sizes[1])
    for _ in range(12):
        number = rng.integers(sizes[0], sizes[1] + 1, 64)
        order = rng.permutation(np.repeat(np.arange(64), number)).astype(np.int32)
        v = rng.normal(0, 1, order.size)
        t = lambda x: torch.as_tensor(x, device=gpu)  # noqa: E731
        r = analysis.order_stats(t(order), t(np.ones(order.size)), np.arange(64), value=t(v), sigma=sigma)
        kept = [_clip(v[order == k], sigma) for k in range(64)]
        assert r['n_kept'].tolist() == [x.size for x in kept]
        for k, x in enumerate(kept):
            if x.size:
                assert r['median'][k] == np.median(x)
                assert abs(r['mean'][k] - np.mean(x)) < 8e-15 and abs(r['std'][k] - np.std(x)) < 8e-15
