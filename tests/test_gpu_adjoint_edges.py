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
