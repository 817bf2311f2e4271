"""The default tiles of a batch are those of handing tiles out one by one to
the variant with the largest, found in no more steps than there are variants."""
import heapq

import numpy as np
import pytest

from marxs_amd import batch


def _one_by_one(n, costs, workgroups):
    load = np.asarray(n, dtype=float) * costs
    k = np.ones(len(load), dtype=np.int64)
    busy = np.flatnonzero(load > 0)
    for _ in range(workgroups - len(busy) if len(busy) else 0):
        k[busy[np.argmax(load[busy] / k[busy])]] += 1
    per = -(-np.asarray(n, dtype=np.int64) // k)
    return np.maximum(64, (per + 63) // 64 * 64)


@pytest.mark.parametrize('workgroups', [1, 16, 256, 1024])
def test_tiles_and_steps(workgroups, monkeypatch):
    rng = np.random.default_rng(workgroups)
    steps = []

    class Counting:
        heapify = staticmethod(heapq.heapify)

        @staticmethod
        def heapreplace(heap, item):
            steps.append(item)
            return heapq.heapreplace(heap, item)
    monkeypatch.setattr(batch, 'heapq', Counting)
    lists = [[100000] * 16, [200000] * 64, [1], [0, 0], [0, 5, 0], [10 ** 6, 1, 77, 10 ** 4], [64] * 300]
    lists += [rng.integers(0, 10 ** 6, size) for size in (2, 3, 7, 16, 64, 200, 256, 300)]
    for n in lists:
        for costs in (np.ones(len(n)), 1. + rng.random(len(n)), np.exp(rng.normal(0, 2, len(n)))):
            steps.clear()
            got = batch._even_tiles(n, costs, workgroups)
            assert len(steps) <= len(n)
            assert np.array_equal(got, _one_by_one(n, costs, workgroups))
