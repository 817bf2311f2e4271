"""Tiles of a batch: about one per workgroup, each variant covered."""
import numpy as np
import pytest

from marxs_amd.batch import _even_tiles


@pytest.mark.parametrize('n', [[100000] * 16, [1], [0, 5, 0], [3001, 3001], [10 ** 6, 1, 77, 10 ** 4],
                               [64] * 300, list(range(1, 40))])
@pytest.mark.parametrize('workgroups', [1, 256])
def test_even_tiles(n, workgroups):
    costs = 1. + np.arange(len(n)) % 3
    tp = _even_tiles(n, costs, workgroups)
    assert tp.shape == (len(n),) and np.all(tp >= 64) and np.all(tp % 64 == 0)
    tiles = -(-np.array(n) // tp)
    # one each at least, no more than the workgroups unless the variants are
    assert np.all((tiles >= 1) == (np.array(n) > 0))
    assert tiles.sum() <= max(workgroups, np.count_nonzero(n))


@pytest.mark.gpu
@pytest.mark.parametrize('prec', [64, 32])
def test_default_tiles_of_a_batch(prec):
    import torch
    from marxs_amd import configs
    from marxs_amd.batch import BatchedTrace
    from marxs_amd.tracer import CompiledInstrument
    from test_gpu_launch_shapes import _columns, _launch, _same, _source
    cis = [CompiledInstrument(configs.cat_rowland_instrument(k)[0]) for k in (60, 150, 90)]
    src = [_source(k, seed=k) for k in (1, 70001, 4097)]
    u = [ci.draw_uniforms(s.n) for ci, s in zip(cis, src)]
    bt = BatchedTrace(cis, src, u, precision=prec)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert bt.plan['n_tiles'] <= cus
    st = bt.run()
    assert len(st) == 3
    for ci, s, k, out in zip(cis, src, u, bt.outputs):
        ref, _ = _launch(ci, s, k, prec)
        got = _columns(out)
        if prec == 64:
            _same(ref, got)
        else:
            for name in ref:
                if ref[name].dtype == torch.int32:
                    assert torch.equal(ref[name], got[name]), name
