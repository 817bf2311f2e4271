"""The fused loss and gradient (mx_adjoint_step) at the edges of what it is
called with (needs an MI355X)."""
import numpy as np
import pytest

from tests.test_gpu_adjoint_step import _problem, _unordered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', [64, 32])
def test_no_photon_with_weight(gpu, precision):
    """No centroid exists: NaN loss and gradients, as the unordered kernels
    give, from the call, the launch and every replay of a graph."""
    import torch
    prob = _problem(gpu, 50, np.full(50, 4), 5)
    prob.weight.zero_()
    loss, gt, gp = prob.loss_and_grad(prob.theta0, prob.period0, precision)
    assert gt.shape == (50, 6) and gp.shape == (50,)
    for x in (loss, gt, gp, *_unordered(prob, prob.theta0, prob.period0, precision)[:2]):
        assert bool(torch.isnan(x).all())
    graph = prob.capture(precision)
    for _ in range(3):
        prob.buffers['loss'].zero_()
        prob.buffers['grad7'].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert bool(torch.isnan(prob.buffers['loss']).all()) and bool(torch.isnan(prob.buffers['grad7']).all())
        assert bool((prob.buffers['moments'] == 0).all())


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('call', ['loss_and_grad', 'launch', 'graph'])
def test_sums_are_in_the_buffers(gpu, precision, call):
    """buffers['sums'] and ['moments'] are those of the unordered kernels, up
    to the order of the sums: 1e-12 of each column's largest value (20 photons
    a facet; a sum of 20 terms differs by 20 * 1.1e-16 of its largest partial
    sums at most, which exceed the largest sum by less than a hundredfold)."""
    import torch
    prob = _problem(gpu, 50, np.full(50, 20), 6)
    pb = prob.buffers
    _unordered(prob, prob.theta0, prob.period0, precision)
    want, moments = pb['sums'].clone(), pb['moments'].clone()
    pb['accum'].fill_(7.)
    if call == 'loss_and_grad':
        prob.loss_and_grad(prob.theta0, prob.period0, precision)
    else:
        pb['theta'].copy_(prob.theta0)
        pb['period'].copy_(prob.period0)
        if call == 'launch':
            prob.launch_loss_and_grad(precision)
        else:
            graph = prob.capture(precision)
            pb['accum'].fill_(7.)
            graph.replay()
        torch.cuda.synchronize()
    assert bool((torch.abs(pb['sums'] - want) <= 1e-12 * torch.abs(want).max(0).values).all())
    assert abs(float(pb['moments'][0] / moments[0]) - 1.) <= 1e-14
    assert abs(float(pb['moments'][2] / moments[2]) - 1.) <= 1e-12
