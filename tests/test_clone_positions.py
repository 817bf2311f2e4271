"""DevicePhotons.clone copies positions whoever wrote them: the caller in
place, a copy that shares them, or a launch that does not go through the
methods that wait for it."""
import copy

import numpy as np
import pytest
import torch

from marxs_amd.tracer import DevicePhotons

N = 1003


def _without_positions():
    rng = np.random.default_rng(2)
    return DevicePhotons(rng.normal(size=(3, N)), rng.normal(size=(3, N)), np.ones(N), np.ones(N), device='cpu')


def _fill(dp):
    dp.pos.copy_(torch.arange(3 * N, dtype=torch.float64).view(3, N))


@pytest.mark.parametrize('how', ['in place', 'assigned', 'kept view', 'shared copy', 'clone of a clone'])
def test_positions_written_by_the_caller(how):
    dp = _without_positions()
    if how == 'in place':
        _fill(dp)
    elif how == 'assigned':
        dp.pos = torch.arange(3 * N, dtype=torch.float64).view(3, N)
    elif how == 'kept view':
        rows = dp.pos[1:]
        dp.clone()
        rows.copy_(torch.arange(2 * N, dtype=torch.float64).view(2, N))
        dp.pos[0] = -1.
    elif how == 'shared copy':
        _fill(copy.copy(dp))
    else:
        dp = dp.clone().clone()
        _fill(dp)
    assert not dp.has_pos or how == 'assigned'
    c = dp.clone()
    assert torch.equal(c.pos, dp.pos) and c.pos.data_ptr() != dp.pos.data_ptr()
    assert c.pos.shape == (3, N) and c.has_pos == dp.has_pos
    c.pos.zero_()
    assert not torch.equal(c.pos, dp.pos)


def test_state_keeps_its_names():
    """A saved photon list holds the columns by the names they are used by."""
    import pickle
    dp = _without_positions()
    _fill(dp)
    state = dp.__reduce_ex__(4)[2]
    assert sorted(state) == ['device', 'dir', 'energy', 'fcols', 'has_pos', 'icols', 'n', 'pol', 'pos', 'prob']
    back = pickle.loads(pickle.dumps(dp))
    assert torch.equal(back.pos, dp.pos) and torch.equal(back.clone().pos, dp.pos)


@pytest.mark.gpu
@pytest.mark.parametrize('graph', [False, True])
def test_positions_of_a_launched_batch(gpu, graph):
    from marxs_amd import configs
    from marxs_amd.batch import BatchedTrace
    from marxs_amd.tracer import CompiledInstrument
    ci = CompiledInstrument(configs.cat_rowland_instrument(50)[0])
    d = torch.zeros((3, N), dtype=torch.float64, device=gpu)
    d[0] = -1.
    pol = torch.zeros_like(d)
    pol[1] = 1.
    one = torch.ones(N, dtype=torch.float64, device=gpu)
    bt = BatchedTrace([ci], [DevicePhotons(d, pol, 0.7 * one, one)], [ci.draw_uniforms(N)], precision=64)
    if graph:
        bt.replay()
    else:
        bt.launch()
    torch.cuda.synchronize()
    out = bt.outputs[0]
    assert bool(torch.isfinite(out.pos).all()) and float(out.pos.abs().max()) > 1.
    assert torch.equal(out.clone().pos, out.pos)
