"""Order statistics at the edges of their bins and chunks (needs an MI355X):
list lengths around the chunk sizes, one and 64 orders, values that repeat,
crowd into one bin, spread over many powers of ten or lie around a large
number, orders that the sample of bin edges misses, and the clipping
parameters.  Counts, kept counts and medians equal numpy's; probability sums,
means and standard deviations equal extended-precision sums over the kept
values to 1e-12 (n values add up to a rounding error of a few times log2(n)
units of 1.1e-16, the deviations from a value of the order to about as many)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clipped(x, sigma, maxiters):
    """Median and the kept values of the oracle's clipping rounds, spreads in
    extended precision."""
    x = x[np.isfinite(x)]
    for _ in range(maxiters):
        if x.size == 0:
            break
        cen = np.median(x)
        sd = float(np.std(x.astype(np.longdouble)))
        keep = x[(x >= cen - sd * sigma) & (x <= cen + sd * sigma)]
        if keep.size == x.size:
            break
        x = keep
    return (np.median(x) if x.size else np.nan), x


def _check(gpu, order, value, prob, orders, res_filter=False, sigma=3., maxiters=5):
    import torch
    from marxs_amd.analysis import order_stats
    t = [torch.as_tensor(np.asarray(v), device=gpu) for v in (order.astype(np.int32), prob, value)]
    got = order_stats(t[0], t[1], orders, value=t[2], res_filter=res_filter, sigma=sigma, maxiters=maxiters)
    again = order_stats(t[0], t[1], orders, value=t[2], res_filter=res_filter, sigma=sigma, maxiters=maxiters)
    for k in got:
        assert np.array_equal(got[k], again[k], equal_nan=True), ('two calls differ', k)
    only = order_stats(t[0], t[1], orders)
    for j, o in enumerate(orders):
        m = order == o
        total = float(prob[m].astype(np.longdouble).sum())
        assert abs(got['prob_sum'][j] - total) <= 1e-12 * total
        assert abs(only['prob_sum'][j] - total) <= 1e-12 * total and only['count'][j] == m.sum()
        c = m & np.isfinite(value) & (prob > 0) if res_filter else m
        assert got['count'][j] == c.sum(), (j, got['count'][j])
        med, kept = _clipped(value[c], sigma, maxiters)
        assert got['n_kept'][j] == kept.size, (j, got['n_kept'][j], kept.size)
        if kept.size == 0:
            assert np.isnan(got['mean'][j]) and np.isnan(got['median'][j]) and np.isnan(got['std'][j])
            continue
        assert got['median'][j] == med, (j, got['median'][j], med)
        wide = kept.astype(np.longdouble)
        sd = float(np.std(wide))
        scale = float(np.abs(kept).max())
        assert abs(got['mean'][j] - float(wide.mean())) <= 1e-12 * sd + 4e-16 * scale, j
        assert abs(got['std'][j] - sd) <= 1e-12 * sd + 4e-16 * scale, (j, got['std'][j], sd)


@pytest.mark.parametrize('n', [1, 2, 63, 2047, 2048, 2049, 4096, 4097, 20000, 150001])
def test_list_lengths(gpu, n):
    rng = np.random.default_rng(n)
    orders = np.arange(-7, 8)
    order = rng.integers(-8, 9, n)
    value = 0.1 * order + 1e-3 * rng.standard_normal(n)
    value[rng.random(n) < 0.02] = rng.choice([np.nan, np.inf, -np.inf, 50.])
    prob = rng.random(n)
    prob[rng.random(n) < 0.1] = 0.
    for res_filter in (False, True):
        _check(gpu, order, value, prob, orders, res_filter)


def _values(kind, n, rng):
    if kind == 'bell':
        return rng.standard_normal(n)
    if kind == 'around_1e9':
        return 1e9 + 1e-3 * rng.standard_normal(n)
    if kind == 'cauchy':
        return rng.standard_cauchy(n)
    if kind == 'constant':
        return np.full(n, 0.1)
    if kind == 'levels':
        return rng.integers(0, 100, n) * 0.3
    if kind == 'atom':
        return np.where(rng.random(n) < 0.5, 0., rng.standard_normal(n))
    if kind == 'line':
        return np.where(rng.random(n) < 0.9, 1.5 + 1e-9 * rng.standard_normal(n), rng.uniform(-10, 10, n))
    if kind == 'powers':
        return rng.choice([-1., 1.], n) * 10. ** rng.uniform(-200, 3, n)
    return np.sort(rng.exponential(size=n))


@pytest.mark.parametrize('kind', ['bell', 'around_1e9', 'cauchy', 'constant', 'levels', 'atom', 'line', 'powers',
                                  'sorted'])
@pytest.mark.parametrize('n, n_orders', [(9001, 1), (60000, 1), (200003, 2), (100003, 64), (2000003, 3)])
def test_distributions(gpu, kind, n, n_orders):
    rng = np.random.default_rng(n + n_orders)
    order = rng.integers(0, n_orders, n)
    _check(gpu, order, _values(kind, n, rng), rng.random(n), np.arange(n_orders))


@pytest.mark.parametrize('sigma, maxiters', [(1., 5), (3., 0), (3., 1), (2., 30), (0.01, 3), (-1., 5), (np.nan, 5)])
@pytest.mark.parametrize('n', [3000, 50000])
def test_clipping_parameters(gpu, sigma, maxiters, n):
    rng = np.random.default_rng(n)
    _check(gpu, rng.integers(0, 2, n), _values('line', n, rng), rng.random(n), np.arange(2), sigma=sigma,
           maxiters=maxiters)


@pytest.mark.parametrize('few', [1, 12, 3000, 30000])
def test_order_missing_from_the_sample(gpu, few):
    """The sample takes one photon of each of 4096 equal parts of the list, at
    a fixed place; the second order's photons all lie elsewhere."""
    n, parts = 4096 * 64, 4096
    i = np.arange(parts, dtype=np.int64)
    b, e = i * n // parts, (i + 1) * n // parts
    taken = b + (((i * 2654435761) & 0xffffffff) >> 7) % (e - b)
    rng = np.random.default_rng(few)
    order = np.zeros(n, dtype=np.int64)
    free = np.setdiff1d(np.arange(n), taken)
    order[rng.choice(free, few, replace=False)] = 1
    value = np.where(order == 1, 1e6 + 1e-3 * rng.standard_normal(n), rng.standard_normal(n))
    _check(gpu, order, value, rng.random(n), np.arange(2))


def test_orders_far_apart_and_sparse(gpu):
    rng = np.random.default_rng(3)
    orders = np.array([-100000, 7, 3, 2 ** 30, 0])
    order = rng.choice(np.append(orders, [1, 2]), 30000)
    _check(gpu, order, rng.standard_normal(30000), rng.random(30000), orders)
