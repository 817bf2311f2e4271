"""Order statistics of lists sorted by order and value, forwards and backwards,
and of lists in runs (needs an MI355X): the figures of the shuffled list, in
about its time.  Counts, kept counts and medians do not depend on the order of
the photons; sums of n values differ by a few times log2(n) units of 1.1e-16,
1e-13 allowed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lists(gpu, n, orders, seed=1):
    import torch
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    order = torch.randint(0, orders, (n,), device=gpu, generator=g, dtype=torch.int32)
    value = torch.randn(n, dtype=torch.float64, device=gpu, generator=g) + order
    prob = torch.rand(n, dtype=torch.float64, device=gpu, generator=g)
    by_value = torch.argsort(value)
    by_both = by_value[torch.argsort(order[by_value], stable=True)]
    runs = torch.arange(n, device=gpu).roll(n // 3)[by_both]
    return order, value, prob, {'shuffled': torch.arange(n, device=gpu), 'sorted': by_both,
                                'backwards': by_both.flip(0), 'by value': by_value, 'runs': runs}


@pytest.mark.parametrize('n', [1, 64, 2047, 2049, 63 * 2048 + 5, 2000000 - 1, 2000000 + 6143])
@pytest.mark.parametrize('orders', [1, 5])
def test_any_order_of_the_photons(gpu, n, orders):
    from marxs_amd.analysis import order_stats
    order, value, prob, lists = _lists(gpu, n, orders)
    want = None
    for name, i in lists.items():
        got = order_stats(order[i], prob[i], np.arange(orders), value=value[i])
        only = order_stats(order[i], prob[i], np.arange(orders))
        if want is None:
            want = got
        for k in ('count', 'n_kept', 'median'):
            assert np.array_equal(got[k], want[k], equal_nan=True), (name, k)
        assert np.array_equal(only['count'], want['count'])
        for k, x in (('prob_sum', got), ('prob_sum', only), ('mean', got), ('std', got)):
            assert np.allclose(x[k], want[k], rtol=1e-13, atol=1e-13, equal_nan=True), (name, k)


def test_time_of_sorted_lists(gpu):
    """Sorting the list changes which bins are looked into and how their
    values lie, within a factor of 3 (measured: 0.8 to 1.1; 4.9 with chunks of
    consecutive photons)."""
    import torch
    from marxs_amd.analysis import order_stats
    order, value, prob, lists = _lists(gpu, 10_000_000, 2)
    best = {}
    for name in ('shuffled', 'sorted', 'backwards'):
        i = lists[name]
        o, v, p = order[i], value[i], prob[i]
        times = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            order_stats(o, p, np.arange(2), value=v)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        best[name] = min(times)
    assert max(best['sorted'], best['backwards']) <= 3. * best['shuffled'], best
