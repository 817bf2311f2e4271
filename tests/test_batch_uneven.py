"""Default tiles of uneven batches: no workgroup is left with a tile of several
times the mean load, whether there are more variants than workgroups or one
list is much longer than the others; even batches keep one tile per workgroup."""
import numpy as np
import pytest

from marxs_amd.batch import _default_tiles, _even_tiles

RNG = np.random.default_rng(0)
UNEVEN = {'one long list of 400': [10 ** 6] + [2000] * 399, 'one long list of 250': [10 ** 6] + [5000] * 249,
          'two decades': (40000 * 10 ** (-2 * RNG.random(300))).astype(int) + 1, 'more than workgroups': [40000] * 300,
          'a few long of many': [300000] * 20 + [3000] * 230, 'all in one': [0] * 255 + [10 ** 6]}


@pytest.mark.parametrize('name', UNEVEN)
@pytest.mark.parametrize('block', [768, 1024])
@pytest.mark.parametrize('spread', [0., 1.])
def test_no_tile_far_above_the_mean(name, block, spread):
    n = np.array(UNEVEN[name])
    costs = np.exp(spread * np.random.default_rng(1).random(len(n)))
    tp = _default_tiles(n, costs, 256, block)
    assert tp.shape == n.shape and np.all(tp >= 64) and np.all(tp % 64 == 0) and np.all(tp < 2 ** 31)
    mean = (n * costs).sum() / 256
    tile = np.minimum(tp, n)
    assert np.all((tile * costs <= 1.6 * mean) | (tile <= block))
    # the longest time that list scheduling can take
    assert mean + (tile * costs).max() <= 2.6 * mean
    # a quarter of the mean or a block: no more tiles than that makes
    assert (-(-n // tp)).sum() <= 256 * 4 + 2 * len(n) + n.sum() // block


@pytest.mark.parametrize('n', [[100000] * 16, [200000] * 64, [3000] * 5, [1], [77, 10 ** 5]])
def test_even_batches(n):
    costs = np.ones(len(n))
    assert np.array_equal(_default_tiles(n, costs, 256, 1024), _even_tiles(n, costs, 256))


def test_blocks_where_they_suffice():
    """1500 photons of a cheap variant beside dearer ones are two blocks, not a
    block and a rest in one tile; and nothing breaks without photons or cost."""
    n = [1500] * 60 + [830] * 60
    tp = _default_tiles(n, np.array([1.] * 60 + [3.] * 60), 256, 768)
    assert np.all(np.minimum(tp, n) <= 768)
    for n, costs in (([0, 0], [1., 1.]), ([5, 0], [0., 0.]), ([10 ** 6] * 300, [0.] * 300)):
        tp = _default_tiles(n, np.array(costs), 256, 768)
        assert np.all(tp >= 64) and np.all(tp < 2 ** 31)
