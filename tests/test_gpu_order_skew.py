"""Order statistics where a few orders hold most photons and have their bins in
proportion (needs an MI355X): one, two or three large orders at any place of
the list of orders, from lists shorter than the sample to several chunks per
workgroup, with values that are not counted, with order numbers that the sample
counts together, and lists just below and above the line.  Bounds as in
test_gpu_order_bins."""
import numpy as np
import pytest

from tests.test_gpu_order_bins import _check

pytestmark = pytest.mark.gpu


def _photons(n, orders, share, seed, spoil=0.):
    """``share``: of the photons, by index into ``orders``; the rest evenly."""
    rng = np.random.default_rng(seed)
    p = np.full(len(orders), (1. - sum(share.values())) / len(orders))
    for k, x in share.items():
        p[k] += x
    order = rng.choice(orders, n, p=p).astype(np.int64)
    value = rng.normal(0, 1, n) * (1. + (order % 3)) + order * 0.1
    value[rng.random(n) < 1e-3] *= 50.
    value[rng.random(n) < spoil] = np.nan
    prob = np.where(rng.random(n) < spoil, 0., rng.random(n))
    return order, value, prob


@pytest.mark.parametrize('n', [3, 100, 4095, 5001, 150001])
@pytest.mark.parametrize('count, share', [(5, {4: .9}), (6, {0: .97}), (15, {7: .6}), (21, {10: .8}), (33, {32: .5, 3: .3}),
                                          (64, {0: .97}), (64, {63: .3, 31: .3, 1: .3}), (64, {5: 1.})])
def test_large_orders(gpu, n, count, share):
    orders = np.arange(-(count // 2), count - count // 2)
    order, value, prob = _photons(n, orders, share, n + count)
    _check(gpu, order, value, prob, orders)


@pytest.mark.parametrize('n', [2000000 + 77, 5000000])
@pytest.mark.parametrize('count, share', [(21, {10: .95}), (64, {40: .97})])
def test_large_orders_of_long_lists(gpu, n, count, share):
    orders = np.arange(count)
    order, value, prob = _photons(n, orders, share, count)
    _check(gpu, order, value, prob, orders)


@pytest.mark.parametrize('share', [.1, .24, .26, .28, .3, .35])
def test_around_the_line(gpu, share):
    orders = np.arange(-12, 3)
    order, value, prob = _photons(60000, orders, {6: share}, int(100 * share))
    _check(gpu, order, value, prob, orders)


@pytest.mark.parametrize('orders', [np.arange(7) * 256, np.array([5, 261, -251, 9, 10, 11]), np.arange(40) * 1000003])
def test_order_numbers_counted_together(gpu, orders):
    order, value, prob = _photons(80000, orders, {1: .7}, 3)
    _check(gpu, order, value, prob, orders)


@pytest.mark.parametrize('res_filter', [False, True])
def test_values_that_are_not_counted(gpu, res_filter):
    orders = np.arange(30)
    order, value, prob = _photons(90000, orders, {12: .9}, 5, spoil=.3)
    _check(gpu, order, value, prob, orders, res_filter=res_filter)
    # the large order is not asked for, or holds nothing that counts
    _check(gpu, order, value, prob, np.delete(orders, 12), res_filter=res_filter)
    value[order == 12] = np.nan
    _check(gpu, order, value, prob, orders, res_filter=res_filter)


def test_time_of_one_large_order(gpu):
    """97 % of the photons in one of 64 orders take at most 3 times as long as
    evenly spread ones (measured: 1.2; 12 with as many bins for each)."""
    import torch
    from marxs_amd.analysis import order_stats
    n = 10_000_000
    g = torch.Generator(device=gpu)
    g.manual_seed(2)
    order = torch.randint(0, 64, (n,), device=gpu, generator=g, dtype=torch.int32)
    value = torch.randn(n, dtype=torch.float64, device=gpu, generator=g)
    prob = torch.rand(n, dtype=torch.float64, device=gpu, generator=g)
    large = torch.where(prob < 0.97, torch.full_like(order, 20), order)
    best = []
    for o in (order, large):
        times = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            order_stats(o, prob, np.arange(64), value=value)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        best.append(min(times))
    assert best[1] <= 3. * best[0], best
