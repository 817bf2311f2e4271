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


@pytest.mark.parametrize('precision', [64, 32])
def test_tasks_outside_the_lists(gpu, precision):
    """A task whose facet or photons there are not counts nothing: the result
    is that of a list in which it is empty, bit for bit."""
    import torch
    prob = _problem(gpu, 50, np.full(50, 300), 7)
    task, src = prob.buffers['task'], prob.buffers['src']
    kept, n = task.clone(), src['n']
    bad = {3: (-1, 0, 100), 10: (50, 0, 100), 20: (2 ** 31 - 1, 5, 6), 30: (7, -1, 100), 40: (7, n - 1, n + 1),
           50: (7, n, n + 128), 60: (7, -2 ** 31, 2 ** 31 - 1), 70: (7, 100, 99)}
    got = []
    for rows in ({j: (0, 0, 0) for j in bad}, bad):
        task.copy_(kept)
        for j, row in rows.items():
            task[j] = torch.tensor(row, dtype=torch.int32)
        prob.buffers['part'].fill_(float('nan'))
        got.append(prob.loss_and_grad(prob.theta0, prob.period0, precision))
    for a, b in zip(*got):
        assert torch.equal(a, b) and bool(torch.isfinite(a).all())


@pytest.mark.parametrize('first', ['launch', 'current', 'graph'])
def test_first_step_on_another_stream(gpu, monkeypatch, first):
    """The kernels that fill the buffers (delayed here) have run when a step
    is launched on another stream than theirs."""
    import torch
    from marxs_amd.adjoint import AdjointProblem
    prob = _problem(gpu, 50, np.full(50, 20), 8)
    want = prob.loss_and_grad(prob.theta0, prob.period0, 64)
    prob._pb = None
    theta, period = prob.theta0.clone(), prob.period0.clone()
    torch.cuda.synchronize()
    tasks = AdjointProblem._tasks

    def delayed(self, *args):
        torch.cuda._sleep(20_000_000)
        return tasks(self, *args)
    monkeypatch.setattr(AdjointProblem, '_tasks', delayed)
    pb = prob._pose_buffers()
    filled = pb['built'][1]
    assert not filled.query()
    other = torch.cuda.Stream()
    if first == 'current':
        with torch.cuda.stream(other):
            got = prob.loss_and_grad(theta, period, 64)
        assert filled.query()
    else:
        with torch.cuda.stream(other):
            pb['theta'].copy_(theta)
            pb['period'].copy_(period)
        if first == 'graph':
            graph = prob.capture(64)
            for _ in range(3):
                pb['loss'].zero_()
                graph.replay()
        else:
            prob.launch_loss_and_grad(64, other.cuda_stream)
        assert filled.query()
        torch.cuda.synchronize()
        got = pb['loss'][0], pb['grad7'][:, :6], pb['grad7'][:, 6]
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert pb['built'] is None


def test_base_pose_in_other_layouts(gpu):
    """The base pose may be a strided view or of single precision: the moments
    are shifted by the same coordinate."""
    import torch
    prob = _problem(gpu, 50, np.full(50, 20), 9)
    theta0, period0 = prob.theta0.to(torch.float32).to(torch.float64), prob.period0.to(torch.float32).to(torch.float64)
    wide = torch.full((50, 12), 3., dtype=torch.float64, device=gpu)
    wide[:, ::2] = theta0
    shifts = []
    for theta, period in ((theta0, period0), (wide[:, ::2], period0.repeat_interleave(2)[::2]),
                          (theta0.to(torch.float32), period0.to(torch.float32))):
        prob.theta0, prob.period0, prob._pb = theta, period, None
        prob.buffers
        shifts.append(prob.y_shift)
    assert shifts[0] == shifts[1] == shifts[2] and np.isfinite(shifts[0])


@pytest.mark.parametrize('precision', [64, 32])
@pytest.mark.parametrize('facets', [2300, 2400])
def test_many_facets(gpu, facets, precision, monkeypatch):
    """Below and above the number of facets and tasks (2300 x 2479, 2400 x
    2587) from which on the moments are added by a kernel of their own; bounds
    as for the smaller problems (sums of 10 photons a facet, moments of 24000)."""
    import torch
    from marxs_amd import configs
    whole = configs.cat_rowland_instrument

    def small_facets(n):
        inst, parts = whole(50)
        gas = configs._gas_with_n(parts['rowland'], n, [301.5, 562.5], [8., 8.],
                                  {'zoom': [1, 3., 3.], 'd': 2e-4, 'order_selector': parts['efficiency']})
        return inst, {**parts, 'gratings': gas}
    monkeypatch.setattr(configs, 'cat_rowland_instrument', small_facets)
    prob = _problem(gpu, facets, np.full(facets, 10), facets)
    assert (facets * prob.buffers['task'].shape[0] >= 6000000) == (facets == 2400)
    loss, gt, gp = prob.loss_and_grad(prob.theta0, prob.period0, precision)
    again = prob.loss_and_grad(prob.theta0, prob.period0, precision)
    assert torch.equal(loss, again[0]) and torch.equal(gt, again[1]) and torch.equal(gp, again[2])
    moments = prob.buffers['moments'].clone()
    loss_u, g7, _ = _unordered(prob, prob.theta0, prob.period0, precision)
    assert abs(loss.item() - loss_u.item()) <= 1e-12 * abs(loss_u.item())
    assert abs(float(moments[2] / prob.buffers['moments'][2]) - 1.) <= 1e-12
    got = torch.cat([gt, gp[:, None]], 1)
    assert bool((torch.abs(got - g7) <= 1e-11 * torch.abs(g7).max(0).values).all())
